"""The runtime on the caller's stream, the default (NULL) stream included:
eager passes and graph replays give the same bits on every stream, after a
change of stream, and from two threads with a model each.  Work on the
default stream is ordered with torch's there, so no synchronisation stands
between a model call and the torch work around it."""
import threading

import pytest
import torch

from servoflow_amd import rdt as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def build(batch, seed=7, int8=0):
    c = R.default_config(layers=2, lang_max=40, img_len=72, batch=batch, int8_weights=int8)
    m = R.RdtModel(c)
    m.init_random(seed, 0.02)
    g = torch.Generator(device=DEV).manual_seed(seed)
    bf = dict(device=DEV, generator=g, dtype=torch.bfloat16)
    m.set_condition(torch.randn(batch, 40, c.hidden, **bf), torch.full((batch,), 33, device=DEV, dtype=torch.int32),
                    torch.randn(batch, 72, c.hidden, **bf), torch.randn(batch, c.hidden, **bf))
    return m, torch.randn(batch, c.horizon, c.action_dim, device=DEV, generator=g)


def passes(m, noise, n=3):
    """Eager then replayed samples, torch work in between on the same stream."""
    outs = [m.sample(noise.clone(), use_graph=False)]
    for i in range(n):
        x = noise * 2.0 - noise
        outs.append(m.sample(x) + 0.0)
        noise = noise + torch.zeros_like(noise)
    return outs


@pytest.mark.parametrize("batch", [1, 3, 10])   # bf16 and fp16 fragment-ordered steps, library step
def test_every_stream_gives_the_same_bits(batch):
    m, noise = build(batch)
    want = m.sample(noise.clone(), use_graph=False)
    side = torch.cuda.Stream()
    for _ in range(2):
        for got in passes(m, noise):
            assert torch.equal(got, want)
        side.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(side):
            outs = passes(m, noise)
        torch.cuda.default_stream().wait_stream(side)
        for got in outs:
            assert torch.equal(got, want)


def test_two_threads_on_the_default_stream():
    models = [build(1, 11), build(3, 12)]
    want = [m.sample(x.clone(), use_graph=False) for m, x in models]
    torch.cuda.synchronize()
    res = [None, None]

    def work(i):
        res[i] = passes(*models[i], n=5)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for i in range(2):
        assert res[i] is not None
        for got in res[i]:
            assert torch.equal(got, want[i])


@pytest.mark.parametrize("batch,int8", [(1, 0), (1, 1), (3, 0), (10, 0)])
def test_first_pass_recorded_by_the_caller(batch, int8):
    """A caller may record a model's first pass into a graph of its own.  The
    weight copies that this pass writes exist only once the graph has run: an
    eager pass before that, and one in between the replays, gives the model's
    result, and so does every replay."""
    print("first pass recorded", batch, int8, flush=True)
    m, noise = build(batch, int8=int8)
    ref, _ = build(batch, int8=int8)
    want = ref.denoise_step(noise, 0.5)
    m.pv_exact(0)   # the condition's P.V forms are known: nothing left to wait for
    torch.cuda.synchronize()
    graph, v = torch.cuda.CUDAGraph(), torch.zeros_like(noise)
    with torch.cuda.graph(graph):
        m.denoise_step(noise, 0.5, out=v)
    assert torch.equal(m.denoise_step(noise, 0.5), want)
    for _ in range(3):
        v.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(v, want)
        assert torch.equal(m.denoise_step(noise, 0.5), want)
