"""Calls of one thread while another thread records a graph: a hoisted
evaluation whose temporaries go beyond the context's arena for the first time,
and the first decode of a level, succeed and leave the recording whole."""
import threading

import numpy as np
import pytest

import _orc
from gpu_util import N, config4, dev, host, uniform_limbs, zeros

pytestmark = pytest.mark.gpu


@pytest.fixture()
def chain():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    import cheddar_amd as chd
    main, aux, _ = config4()
    main = main[:6]
    ctx = chd.Context(chd.Param(main, aux, [(i, 0) for i in range(1, 7)]))
    return chd, ctx, main, aux


def _beside_a_capture(chd, main, mode, call):
    """call() on a thread of its own while this one records two transforms;
    returns its result when the recording replays to the oracle's words"""
    import torch
    r = np.random.default_rng(0xCA97)
    a = uniform_limbs(r, main[:2])
    want = _orc.ntt_batch(a.reshape(-1), 16, main[:2]).reshape(2, N)
    plan = chd.NttPlan(main[:2])
    src, dst = dev(a), zeros(2, N)
    plan.forward(dst, src, 2)
    torch.cuda.synchronize()
    out = []

    def work():
        try:
            out.append(call())
        except Exception as e:
            out.append(e)
    # private stream and explicit ends: a failed recording must not stay open
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(stream):
        graph.capture_begin(capture_error_mode=mode)
        plan.forward(dst, src, 2)
        t = threading.Thread(target=work)
        t.start()
        t.join()
        graph.capture_end()
    torch.cuda.synchronize()
    assert not isinstance(out[0], Exception), out[0]
    for _ in range(3):
        dst.zero_()
        graph.replay()
        assert np.array_equal(host(dst), want)
    return out[0]


def test_added_chunk_beside_a_capture(chain):
    import torch
    chd, ctx, main, aux = chain
    r = np.random.default_rng(0xCA98)
    L, level = 5, 4
    key = tuple([dev(uniform_limbs(r, main + aux))] for _ in range(2))

    def handle(ngs):
        h = chd.Hoist(ctx, level, [2 * k for k in range(ngs)], [0, 1],
                      {(2 * k, b): dev(uniform_limbs(r, main[:L] + aux))
                       for k in range(ngs) for b in range(2)})
        return h, {rot: key for rot in h.required_rotations()}
    small, large = handle(1), handle(14)
    x = (dev(uniform_limbs(r, main[:L])), dev(uniform_limbs(r, main[:L])))
    res = (zeros(L - 1, N), zeros(L - 1, N))
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    # leaves the baby steps' memory in the pool
    small[0].run(res, x, small[1], stream=side.cuda_stream)
    torch.cuda.synchronize()
    del small
    _beside_a_capture(chd, main, "global", lambda: large[0].run(
        res, x, large[1], stream=side.cuda_stream))
    got = [host(t) for t in res]
    large[0].run(res, x, large[1], stream=side.cuda_stream)
    for t, w in zip(res, got):
        assert np.array_equal(host(t), w)

def test_first_decode_beside_a_capture(chain):
    import torch
    chd, ctx, main, aux = chain
    r = np.random.default_rng(0xCA99)
    msg = r.normal(size=512) + 1j * r.normal(size=512)
    pt = zeros(5, N)
    stream = torch.cuda.Stream().cuda_stream
    torch.cuda.synchronize()
    slots = ctx.encode(4, 0, float(1 << 30), msg, pt, stream)
    got = _beside_a_capture(
        chd, main, "thread_local",
        lambda: ctx.decode(4, float(1 << 30), slots, pt, stream))
    assert np.abs(got - msg).max() < 1e-5
    assert np.array_equal(ctx.decode(4, float(1 << 30), slots, pt, stream),
                          got)
