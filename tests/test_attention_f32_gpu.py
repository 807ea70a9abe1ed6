"""The fp32 attention kernel deals 16-key blocks to four waves and merges their
shares: key counts around the block and the round of four (waves without a
key), split or not, with length and causal masks, against float64.

Bound: a score is a 64-term fp32 dot product of N(0, 1) rows, scaled by 1/8:
error below 64 * 2^-24 * sum|q_i k_i| / 8 < 64 * 2^-24 * 64 / 8 * 2 (rows of
64 with mean |q k| 0.64, twice that for the largest) = 6.1e-5 relative on a
weight, and on outputs of at most 5: 1e-4 for rounding that does not all add
up the same way."""
import pytest
import torch

from servoflow_amd.attention import attention

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(q, k, v, keep):
    s = (q.double() @ k.double().transpose(-1, -2)) / 8.0
    s = s.masked_fill(~keep, float("-inf"))
    p = torch.softmax(s, -1).nan_to_num(0.0)   # no key kept: zeros
    return p @ v.double()


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("Sk", [1, 15, 16, 17, 48, 63, 64, 65, 80, 129, 300])
def test_key_counts_and_masks(Sk, splits):
    B, H, Sq = 2, 3, 37
    g = torch.Generator(device=DEV).manual_seed(Sk)
    q, k, v = (torch.randn(B, H, n, 64, device=DEV, generator=g) for n in (Sq, Sk, Sk))
    vl = torch.tensor([max(1, Sk - 1), (Sk + 1) // 2], device=DEV, dtype=torch.int32)
    keep = torch.ones(B, 1, Sq, Sk, dtype=torch.bool, device=DEV)
    cols = torch.arange(Sk, device=DEV)
    lens = cols[None, None, None, :] < vl[:, None, None, None]
    print("fp32 attention", Sk, splits, flush=True)
    for kw, kp in (({}, keep), ({"valid_len": vl}, keep & lens),
                   ({"is_causal": True}, keep & (cols[None, :] <= torch.arange(Sq, device=DEV)[:, None]))):
        got = attention(q, k, v, out_dtype=torch.float32, num_splits=splits, **kw).double()
        assert (got - reference(q, k, v, kp)).abs().max().item() <= 1e-4, kw


@pytest.mark.parametrize("B,H,Sq,splits", [(1, 1, 1, 1), (1, 7, 67, 1), (1, 8, 16, 1), (2, 8, 67, 2), (3, 5, 33, 3),
                                           (1, 9, 131, 4)])
def test_every_query_block_is_computed_once(B, H, Sq, splits):
    """Groups of (b, h, split) below, at and past multiples of 8, the unit in
    which workgroups are dealt; keys of their own strides in half the cases."""
    Sk = 150
    g = torch.Generator(device=DEV).manual_seed(100 * H + Sq)
    q = torch.randn(B, H, Sq, 64, device=DEV, generator=g)
    k, v = (torch.randn(B, H, Sk, 64, device=DEV, generator=g) for _ in range(2))
    if H % 2:   # [B, S, H, 64] storage
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    keep = torch.ones(B, 1, Sq, Sk, dtype=torch.bool, device=DEV)
    print("fp32 attention grid", B, H, Sq, splits, flush=True)
    got = attention(q, k, v, out_dtype=torch.float32, num_splits=splits).double()
    assert (got - reference(q, k, v, keep)).abs().max().item() <= 1e-4


@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 8, 11, 11), (1, 8, 40, 17), (26, 8, 67, 33), (26, 8, 67, 67), (26, 8, 67, 256), (26, 8, 67, 257),
                                       (103, 8, 67, 17), (103, 8, 67, 256), (103, 8, 67, 257), (147, 7, 67, 50)])
def test_waves_per_workgroup(B, H, Sq, Sk):
    """Both sides of the rule for one, two and four waves: one key block and
    two, 1040 and 4120 workgroups with 16 key blocks and with 17; a full and a
    ragged set of keys, a batch element without a key among them."""
    g = torch.Generator(device=DEV).manual_seed(1000 * B + Sk)
    q, k, v = (torch.randn(B, H, n, 64, device=DEV, generator=g) for n in (Sq, Sk, Sk))
    vl = torch.randint(0, Sk + 1, (B,), device=DEV, generator=g, dtype=torch.int32)
    vl[0] = 0
    keep = torch.ones(B, 1, Sq, Sk, dtype=torch.bool, device=DEV)
    lens = torch.arange(Sk, device=DEV)[None, None, None, :] < vl[:, None, None, None]
    print("fp32 attention waves", B, H, Sq, Sk, flush=True)
    for kw, kp in (({}, keep), ({"valid_len": vl}, keep & lens)):
        ref = reference(q, k, v, kp)
        # a rounding to bf16's 8 bits, to nearest, is at most 2^-8 of the value
        for odt, step in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8)):
            got = attention(q, k, v, out_dtype=odt, **kw).double()
            assert ((got - ref).abs() <= 1e-4 + step * ref.abs()).all(), (odt, list(kw))
