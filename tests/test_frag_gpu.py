"""GPU tests of the fragment-ordered projections (sf_gemm_frag, sf_frag_pack,
sf_norm_frag) and of the attention's fragment-ordered output and fp32 Q rows.

Products of 16-bit operands are exact in fp32, so a projection differs from
the float64 reference by its fp32 summation only: with K <= 8192 terms of
|a w| ~ 0.02 that is below 2e-5 of the result's norm (measured 1e-6).  16-bit
outputs add one rounding to nearest: of 8 (bf16) or 11 (fp16) significant
bits, so at most 2^-8 or 2^-11 of the value."""
import ctypes

import pytest
import torch

from oracle import oracle as O
from servoflow_amd import abi
from servoflow_amd import kernels as K
from servoflow_amd.attention import attention, make_desc, workspace_bytes

pytestmark = pytest.mark.gpu
DEV = "cuda"
_ROUND = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def to_frag(x):
    """Row-major [R, K] 16-bit -> fragment order, rows padded with NaN (no
    result may depend on the padding)."""
    R, Kd = x.shape
    pad = torch.full(((-R) % 16, Kd), float("nan"), dtype=x.dtype, device=x.device)
    return torch.cat([x, pad]).view(-1, 16, Kd // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous().view(-1, Kd)


def from_frag(f, R):
    return f.view(f.shape[0] // 16, f.shape[1] // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(f.shape)[:R]


def i8_frag(q):
    N, Kd = q.shape
    return q.view(N // 16, 16, Kd // 64, 2, 4, 8).permute(0, 2, 4, 1, 3, 5).contiguous().view(N, Kd)


def randn(seed, *shape, dtype=torch.float32, std=1.0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return (torch.randn(*shape, device=DEV, generator=g) * std).to(dtype)


def weights(seed, N, Kd, kind, adt):
    """(fragment-ordered copy, scale or None, float64 values the copy means)."""
    w = randn(seed, N, Kd, std=0.02)
    if kind in ("int8", "codes16"):   # codes16: int8 codes widened to fp16, with their scale
        s = w.abs().amax(1) / 127
        q = torch.clamp(torch.round(w / s[:, None]), -127, 127).to(torch.int8)
        return K.frag_pack([q], [torch.int8 if kind == "int8" else adt])[0], s, q.double() * s.double()[:, None]
    w = w.to(torch.bfloat16)
    return K.frag_pack([w], [adt])[0], None, w.to(adt).double()


def rel(got, ref):
    got, ref = got.double(), ref.double()
    assert torch.isfinite(got).all()
    return ((got - ref).norm() / ref.norm()).item()


def test_pack_layouts():
    w = randn(1, 48, 192, dtype=torch.bfloat16)
    wide = randn(2, 32, 264, dtype=torch.bfloat16)[:, :256]           # row stride 264
    q = torch.randint(-128, 128, (16, 128), dtype=torch.int8, device=DEV)
    a, b, c, d, e = K.frag_pack([w, w, wide, q, q], [torch.bfloat16, torch.float16, torch.bfloat16, torch.int8,
                                                     torch.float16])
    assert torch.equal(e, to_frag(q.to(torch.float16)))
    assert torch.equal(a, to_frag(w)) and torch.equal(b, to_frag(w.to(torch.float16)))
    assert torch.equal(c, to_frag(wide.contiguous())) and torch.equal(d, i8_frag(q))


# every tile of the rule -- row tiles of 2 to 9 blocks with partial last
# blocks, one row; column tiles of 32, 64 and 128, more than 256 of them, a
# count that is no multiple of 8 -- and K of one chunk, of fewer chunks than
# waves x groups, and ragged over the waves
@pytest.mark.parametrize("M,N,Kd", [(67, 2048, 2048), (1, 64, 64), (16, 128, 2048), (134, 2048, 2048), (160, 6144, 192),
                                    (67, 6144, 1088), (81, 96, 320), (33, 32, 4096), (134, 8192, 576), (67, 2048, 8192),
                                    (402, 2048, 320), (539, 2048, 192), (640, 2048, 256), (603, 6144, 2048),
                                    (500, 6144, 448), (1072, 2048, 64), (1000, 2048, 704), (450, 6144, 128),
                                    (700, 4096, 128), (999, 384, 192), (15, 2048, 2048), (19, 2048, 320),
                                    (64, 2048, 192), (65, 1024, 2048), (48, 6144, 128)])
@pytest.mark.parametrize("kind,adt", [("w16", torch.bfloat16), ("w16", torch.float16), ("int8", torch.bfloat16),
                                      ("int8", torch.float16), ("codes16", torch.float16)])
def test_plain(M, N, Kd, kind, adt):
    a, (wf, s, w64) = randn(3, M, Kd, dtype=adt), weights(4, N, Kd, kind, adt)
    b = randn(5, N)
    ref = a.double() @ w64.t() + b.double()
    got = K.gemm_frag(M, to_frag(a), wf, b, w_scale=s)
    assert rel(got, ref) < 2e-5
    x = randn(6, M, N)
    x0 = x.clone()
    K.gemm_frag(M, to_frag(a), wf, b, w_scale=s, out=x, accumulate=True)
    assert torch.equal(x, x0 + got)
    rs = K.gemm_frag(M, to_frag(a), wf, b, w_scale=s, out=torch.empty(M, N + 12, device=DEV)[:, :N])
    assert torch.equal(rs, got)
    h = K.gemm_frag(M, to_frag(a), wf, b, w_scale=s, act=abi.SF_ACT_GELU_TANH, c_frag=True, out_dtype=torch.float16)
    href = 0.5 * ref * (1 + torch.tanh(0.7978845608028654 * (ref + 0.044715 * ref ** 3)))
    assert rel(from_frag(h, M), href) < _ROUND[torch.float16]


@pytest.mark.parametrize("kind,dt,full", [("w16", torch.bfloat16, 160), ("int8", torch.float16, 160),
                                          ("w16", torch.float16, 1072)])
def test_row_does_not_depend_on_the_batch(kind, dt, full):
    a, (wf, s, _) = randn(7, full, 2048, dtype=dt), weights(8, 2048, 2048, kind, dt)
    whole = K.gemm_frag(full, to_frag(a), wf, w_scale=s)
    for M in (1, 17, 67, 134, 402, 804, 1072):
        if M < full:
            assert torch.equal(K.gemm_frag(M, to_frag(a[:M].contiguous()), wf, w_scale=s), whole[:M])


@pytest.mark.parametrize("M,N", [(67, 2048), (134, 2048), (5, 64), (16, 2048), (19, 2048), (49, 2048), (19, 4096), (97, 4096), (640, 2048), (1072, 2048), (402, 1024)])
@pytest.mark.parametrize("kind,adt,ndt", [("w16", torch.bfloat16, torch.bfloat16), ("int8", torch.bfloat16, torch.float16),
                                          ("w16", torch.float16, torch.float16), ("codes16", torch.float16, torch.float16)])
def test_add_norm_and_its_consumer(M, N, kind, adt, ndt):
    """The deferred pair: x * gamma and tile sums out of one projection, the
    row scale applied by the next, against the normalised rows' product."""
    a, (wf, s, w64) = randn(9, M, 512, dtype=adt), weights(10, N, 512, kind, adt)
    b, gamma, x = randn(11, N), 1 + randn(12, N, std=0.1), randn(13, M, N)
    xr = x.double() + a.double() @ w64.t() + b.double()
    n, ss = K.gemm_frag_add_norm(M, to_frag(a), wf, b, x, gamma, norm_dtype=ndt, w_scale=s)
    assert rel(x, xr) < 2e-6
    assert rel(ss.sum(1), xr.square().sum(1)) < 2e-6
    assert torch.equal(from_frag(n, M), (x * gamma).to(ndt))
    wf2, _, w2 = weights(14, 256, N, "w16", ndt)
    guard = {"x": x, "x_gamma": gamma} if ndt == torch.float16 else {}
    got = K.gemm_frag(M, n, wf2, b[:256] if N >= 256 else None, row_ss=ss, row_n=N, **guard)
    ref = (from_frag(n, M).double() @ w2.t()) * torch.rsqrt(xr.square().mean(1, keepdim=True) + 1e-6)
    ref = ref + (b[:256].double() if N >= 256 else 0)
    assert rel(got, ref) < 2e-5


@pytest.mark.parametrize("B,S,H", [(1, 67, 32), (2, 67, 32), (3, 11, 2), (1, 160, 1), (1, 19, 32), (1, 32, 32), (1, 4, 32)])
@pytest.mark.parametrize("kind", ["w16", "int8"])
@pytest.mark.parametrize("deferred", [False, True])
def test_heads(B, S, H, kind, deferred):
    """Finished rows, and the rows of a deferred norm: their 1/rms after the product."""
    M, D = B * S, H * 64
    a, (wf, s, w64) = randn(15, M, D, dtype=torch.bfloat16), weights(16, 3 * D, D, kind, torch.bfloat16)
    af, rows, row = to_frag(a), a.double(), {}
    if deferred:
        x = randn(22, M, D) * torch.linspace(0.1, 30, M, device=DEV)[:, None]
        af, ss = K.norm_frag(x, 1 + randn(23, D, std=0.1), out_dtype=torch.bfloat16, deferred=True)
        rows = from_frag(af, M).double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-6)
        row = {"row_ss": ss, "row_n": D}
    b = randn(17, 3 * D)
    gq, gk = 1 + randn(18, 64, std=0.1), 1 + randn(19, 64, std=0.1)
    outs = [torch.full((B, H, S, 64), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(3)]
    K.gemm_frag_heads(M, af, wf, b, S, H, outs, (gq, gk, None), w_scale=s, **row)
    ref = (rows @ w64.t() + b.double()).view(B, S, 3, H, 64).permute(2, 0, 3, 1, 4)
    for j, g in enumerate((gq, gk, None)):
        r = ref[j]
        if g is not None:
            r = r * torch.rsqrt(r.square().mean(-1, keepdim=True) + 1e-6) * g.double()
        assert rel(outs[j], r) < _ROUND[torch.bfloat16]


@pytest.mark.parametrize("rows,cols", [(67, 2048), (1, 64), (160, 4096), (33, 1024), (5, 2112)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_norm_frag(rows, cols, dt):
    x, gamma = randn(20, rows, cols + 4)[:, :cols], 1 + randn(21, cols, std=0.1)
    out, _ = K.norm_frag(x, gamma, out_dtype=dt)
    ref = x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-6) * gamma.double()
    assert rel(from_frag(out, rows), ref) < _ROUND[dt]
    out, ss = K.norm_frag(x, gamma, out_dtype=dt, deferred=True)
    assert torch.equal(from_frag(out, rows), (x * gamma).to(dt))
    assert rel(ss, x.double().view(rows, -1, 64).square().sum(-1)) < 1e-6


@pytest.mark.parametrize("M,N,kind", [(67, 2048, "w16"), (19, 2048, "w16"), (134, 256, "int8"), (81, 4096, "w16"), (160, 2048, "int8"),
                                      (640, 2048, "w16"), (1072, 512, "w16")])
def test_fp16_rows_out_of_range(M, N, kind):
    """Deferred fp16 rows whose x * gamma leaves fp16's range, is far below
    it, or is zero: those rows come from the fp32 residual, normalised first;
    the others are bit for bit what they are without such neighbours."""
    zero, small, big = 0, 7, M - 1
    a = torch.zeros(M, 64, dtype=torch.bfloat16, device=DEV)
    wz = K.frag_pack([torch.zeros(N, 64, dtype=torch.bfloat16, device=DEV)], [torch.bfloat16])[0]
    gamma, x = 1 + randn(40, N, std=0.1), randn(41, M, N)
    plain = x.clone()
    x[zero], x[small], x[big] = 0, x[small] * 1e-6, x[big] * 1e5
    wf, s, w64 = weights(42, 512, N, kind, torch.float16)
    b = randn(43, 512)
    got = []
    for rows in (x, plain):
        n, ss = K.gemm_frag_add_norm(M, to_frag(a), wz, None, rows, gamma, norm_dtype=torch.float16)
        got.append(K.gemm_frag(M, n, wf, b, w_scale=s, row_ss=ss, row_n=N, x=rows, x_gamma=gamma))
        assert (not torch.isfinite(ss[big].sum())) == (rows is x)
    ref = (x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-6) * gamma.double()) @ w64.t() + b.double()
    for r in (zero, small, big, 1):
        assert rel(got[0][r], ref[r]) < _ROUND[torch.float16]
    same = [r for r in range(M) if r not in (zero, small, big)]
    assert torch.equal(got[0][same], got[1][same])


# (x's scale, gamma's scale): x * gamma deep in fp16's subnormals, just above
# and below the mark, x of ordinary size (no better off normalised), and large
@pytest.mark.parametrize("xs,gs", [(0.0042, 0.03), (0.0042, 1e-3), (0.0078, 3e-3), (0.3, 1e-3), (0.9, 2e-4), (0.03, 0.1),
                                   (3.0, 1e-3), (300.0, 3e-3), (1e-4, 40.0)])
@pytest.mark.parametrize("M,N", [(67, 2048), (402, 512)])
@pytest.mark.parametrize("entry", [False, True])
def test_fp16_rows_of_small_products(M, N, entry, xs, gs):
    """Deferred fp16 rows whose x * gamma is small keep the precision of rows
    normalised before their rounding to fp16, from both producers.  A rounding
    to nearest of 11 bits has a relative error below 2^-11, uniformly spread
    below 2^-11 / sqrt(3) of the value; the product's share is that of its
    terms.  The second half of the columns has gamma's scale a hundredth: its x
    is a hundred times larger in every third row, and the first half's zero."""
    gamma, x = (1 + randn(50, N, std=0.1)) * gs, randn(51, M, N) * xs
    gamma[N // 2:] *= 0.01
    x[::3, N // 2:] *= 100
    x[::3, :N // 2] = 0
    wf, s, w64 = weights(52, 512, N, "w16", torch.float16)
    if entry:
        n, ss = K.norm_frag(x, gamma, out_dtype=torch.float16, deferred=True)
    else:
        a = torch.zeros(M, 64, dtype=torch.bfloat16, device=DEV)
        wz = K.frag_pack([torch.zeros(N, 64, dtype=torch.bfloat16, device=DEV)], [torch.bfloat16])[0]
        n, ss = K.gemm_frag_add_norm(M, to_frag(a), wz, None, x, gamma, norm_dtype=torch.float16)
    got = K.gemm_frag(M, n, wf, None, row_ss=ss, row_n=N, x=x, x_gamma=gamma)
    norm = x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-6) * gamma.double()
    ref = norm @ w64.t()
    # what a normalised row's own subnormals (half a step of 2^-24) add
    sub = 2.0 ** -25 / norm.square().mean(1).sqrt()
    err = (got.double() - ref).norm(dim=1) / ref.norm(dim=1)
    bound = 2.0 ** -11 / 3 ** 0.5 + sub
    print("small products", M, N, entry, xs, gs, (err / bound).max().item(), flush=True)
    assert (err < bound).all()


# the one-wave and grouped short-key kernels, the query-block grid, key splits
# with the merge, the unsplit 80-row grid, and fp32 inputs
@pytest.mark.parametrize("B,H,Sq,Sk,dt", [(1, 32, 67, 67, torch.bfloat16), (8, 32, 67, 67, torch.float16),
                                          (2, 3, 41, 700, torch.bfloat16), (1, 32, 67, 4374, torch.bfloat16),
                                          (8, 32, 67, 300, torch.float16), (1, 4, 67, 1500, torch.float32)])
def test_attention_frag_output(B, H, Sq, Sk, dt):
    q, k, v = (randn(22 + i, B, H, s, 64, dtype=dt) for i, s in enumerate((Sq, Sk, Sk)))
    odt = torch.float16 if dt == torch.float16 else torch.bfloat16
    ref = attention(q, k, v, out_dtype=odt).permute(0, 2, 1, 3).reshape(B * Sq, H * 64)
    out = torch.empty((B * Sq + 15) // 16 * 16, H * 64, dtype=odt, device=DEV)
    desc = make_desc(q, k, v, torch.empty(B, H, Sq, 64, dtype=odt, device=DEV))
    desc.o_frag = 1
    ws = torch.empty(max(16, workspace_bytes(desc)), dtype=torch.uint8, device=DEV)
    st = abi.lib().sf_attn_fwd(ctypes.byref(desc), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                               ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert st == abi.SF_OK
    assert torch.equal(from_frag(out, B * Sq), ref)
    desc.out_dtype = abi.SF_F32
    assert abi.lib().sf_attn_fwd(ctypes.byref(desc), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                 ws.data_ptr(), ws.numel(), None) == abi.SF_ENOTSUP


# query blocks, key splits, the unsplit 80-row grid with a partial chunk, keys
# of the short-key kernel (the ring kernel takes them), exact P.V
# and V in bf16 or, as the model's cross-attention caches it, in fp16
@pytest.mark.parametrize("B,H,Sq,Sk,form", [(1, 32, 67, 517, "bf16"), (1, 32, 67, 517, "fp16"), (1, 32, 67, 4374, "bf16"),
                                            (1, 32, 67, 4374, "fp16"), (2, 32, 67, 4374, "exact"), (8, 32, 67, 300, "bf16"),
                                            (8, 32, 67, 300, "fp16"), (1, 4, 133, 2000, "fp16"), (1, 8, 19, 40, "exact"),
                                            (1, 8, 19, 40, "fp16")])
def test_attention_fp32_q_rows(B, H, Sq, Sk, form):
    """Q as fp32 projection rows, normalised on load, against the oracle's
    attention over rows normalised and rounded to bf16 beforehand."""
    exact = form == "exact"
    rows = randn(30, B * Sq, H * 64, std=3.0)
    gamma = 1 + randn(31, 64, std=0.1)
    k, v = (randn(32 + i, B, H, Sk, 64, dtype=torch.bfloat16) for i in range(2))
    if form == "fp16":
        v = v.to(torch.float16)
    q32 = rows.view(B, Sq, H, 64).permute(0, 2, 1, 3)
    r64 = q32.double()
    q = (r64 * torch.rsqrt(r64.square().mean(-1, keepdim=True) + 1e-6) * gamma.double()).to(torch.bfloat16).contiguous()
    out = torch.empty(B, H, Sq, 64, device=DEV)
    desc = make_desc(q, k, v, out, exact_pv=exact, q_gamma=gamma)
    desc.q_rows32 = rows.data_ptr()
    ws = torch.empty(max(16, workspace_bytes(desc)), dtype=torch.uint8, device=DEV)
    st = abi.lib().sf_attn_fwd(ctypes.byref(desc), None, k.data_ptr(), v.data_ptr(), out.data_ptr(), ws.data_ptr(),
                               ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert st == abi.SF_OK
    # a bf16 rounding tie between the fp32 and the float64 norm moves a Q
    # element by 2^-8 of itself, so an output by far less than this
    ref = O.attention_f32(*(t.float().cpu().numpy() for t in (q, k, v)))
    assert rel(out.cpu(), torch.from_numpy(ref)) < 1e-3


def test_refused():
    a, w = torch.zeros(16, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV)
    out = torch.zeros(16, 64, device=DEV)

    def call(**kw):
        d = abi.FragGemmDesc()
        d.M, d.N, d.K, d.A, d.a_dtype, d.W, d.w_dtype = 16, 64, 64, a.data_ptr(), abi.SF_BF16, w.data_ptr(), abi.SF_BF16
        d.epilogue, d.C, d.ldc, d.c_dtype = abi.SF_EPI_PLAIN, out.data_ptr(), 64, abi.SF_F32
        for k, v in kw.items():
            setattr(d, k, v)
        return abi.lib().sf_gemm_frag(ctypes.byref(d), None)

    assert call() == abi.SF_OK
    torch.cuda.synchronize()
    for kw, st in [({"K": 32}, abi.SF_ENOTSUP), ({"N": 16}, abi.SF_ENOTSUP),
                   ({"a_dtype": abi.SF_F32}, abi.SF_ENOTSUP), ({"w_dtype": abi.SF_F16}, abi.SF_ENOTSUP),
                   ({"w_dtype": abi.SF_I8}, abi.SF_EINVAL), ({"ldc": 62}, abi.SF_EINVAL), ({"C": out.data_ptr() + 4}, abi.SF_EINVAL),
                   ({"c_frag": 1}, abi.SF_EINVAL), ({"epilogue": abi.SF_EPI_PARTIALS}, abi.SF_ENOTSUP),
                   ({"a_row_ss": out.data_ptr(), "a_row_tiles": 65, "a_row_n": 64}, abi.SF_EINVAL), ({"act": 3}, abi.SF_EINVAL)]:
        assert call(**kw) == st, kw
    assert call(M=0) == abi.SF_OK


def test_unguarded_fp16_rows_refused():
    """Deferred fp16 rows may have left fp16's range, so they need the fp32
    rows behind them; the per-head epilogue has no guard and takes none."""
    a, w = torch.zeros(16, 64, dtype=torch.float16, device=DEV), torch.zeros(192, 64, dtype=torch.float16, device=DEV)
    ss, x, gamma = torch.ones(16, 1, device=DEV), torch.ones(16, 64, device=DEV), torch.ones(64, device=DEV)
    with pytest.raises(abi.SfError) as e:
        K.gemm_frag(16, a, w, row_ss=ss, row_n=64)
    assert e.value.status == abi.SF_EINVAL
    assert torch.equal(K.gemm_frag(16, a, w, row_ss=ss, row_n=64, x=x, x_gamma=gamma), torch.zeros(16, 192, device=DEV))
    outs = [torch.empty(1, 1, 16, 64, dtype=torch.bfloat16, device=DEV) for _ in range(3)]
    with pytest.raises(abi.SfError) as e:
        K.gemm_frag_heads(16, a, w, None, 16, 1, outs, row_ss=ss, row_n=64)
    assert e.value.status == abi.SF_ENOTSUP
