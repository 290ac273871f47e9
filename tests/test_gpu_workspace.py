"""Calls that need more temporaries than a context's arena holds: the chunks
it adds serve later calls of other sizes and streams, interleaved with calls
inside the arena, with the same results every time."""
import numpy as np
import pytest

from gpu_util import N, config4, dev, host, uniform_limbs, zeros

pytestmark = pytest.mark.gpu


def test_added_chunks_serve_later_calls():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    import cheddar_amd as chd
    main, aux, _ = config4()
    main = main[:6]
    ctx = chd.Context(chd.Param(main, aux, [(i, 0) for i in range(1, 7)]))
    r = np.random.default_rng(0xA2E)
    L, level = 5, 4
    keys = {}

    def handle(ngs, nbs):
        gs = [nbs * k for k in range(ngs)]
        pts = {(g, b): dev(uniform_limbs(r, main[:L] + aux))
               for g in gs for b in range(nbs)}
        h = chd.Hoist(ctx, level, gs, list(range(nbs)), pts)
        for rot in h.required_rotations():
            if rot not in keys:
                keys[rot] = tuple([dev(uniform_limbs(r, main + aux))]
                                  for _ in range(2))
        return h
    # 14 and 6 giant steps: temporaries of several sizes beyond the arena
    hs = [handle(14, 2), handle(6, 3)]
    x = [dev(uniform_limbs(r, main[:L])) for _ in range(4)]
    mult = tuple([dev(uniform_limbs(r, main + aux))] for _ in range(2))

    def run(k, stream):
        res = (zeros(L - 1, N), zeros(L - 1, N))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            if k < 2:
                hs[k].run(res, (x[0], x[1]), keys)
            else:
                ctx.hmult(level, res, (x[0], x[1]), (x[2], x[3]), *mult)
        return res
    main_stream, side = torch.cuda.current_stream(), torch.cuda.Stream()
    want = [[host(t) for t in run(k, main_stream)] for k in range(3)]
    for i in range(4):
        # no synchronisation between the three calls but the workspace's own
        outs = []
        for k in ((0, 1, 2), (1, 2, 0), (2, 0, 1), (1, 0, 2))[i]:
            outs.append((k, run(k, side if (i + k) % 2 else main_stream)))
        for k, out in outs:
            for a, b in zip(out, want[k]):
                assert np.array_equal(host(a), b), (i, k)
