"""Block maps spread on the device (scenes without blocks in a launch, many scenes, one) and the graph
from its second replay on (63 to 97 steps), against each scene's own run, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(amd, sc):
    s = amd.PPPMSolver(sc.res, sc.dl, sc.dt, sc.min_pos, 0, 0.83, sc.c)
    s.set_mesh(sc.verts, sc.tris)
    return s


# mixed variants leave scenes without blocks in some launches, first, last and in between
@pytest.mark.parametrize("edges,variants,steps", [([24], [1], 63), ([24, 37, 30], [0, 2, 0], 64),
                                                  ([24, 37, 30, 26], [1, 0, 3, 4], 65), ([24] * 40, None, 97)])
def test_batch_setup_bitexact(amd, scenes_mod, edges, variants, steps):
    import torch
    sc = [scenes_mod.c3_scene(n, 1 + i % 2, seed=i, steps=steps) for i, n in enumerate(edges)]
    lis = [(3 * x.res // 4 + 2, x.res // 2, x.res // 2) for x in sc]
    acc = [torch.from_numpy(x.neumann[:steps]).cuda() for x in sc]
    hs = [_solver(amd, x) for x in sc]
    b = amd.PPPMBatch(hs)
    if variants is not None:
        b.set_variants(variants)
    out = torch.zeros(steps, len(sc), device="cuda")
    w = torch.randn(steps, len(sc), 1, device="cuda")
    for graph in (True, False):
        for s in hs:
            s.reset()
        b.run(acc, steps, lis, out, use_graph=graph)
        b.adjoint_reset(steps - 1)
        grads = [torch.zeros(steps, s.nt, device="cuda") for s in hs]
        b.adjoint_run(w, steps, [[x] for x in lis], grads, use_graph=graph)
        torch.cuda.synchronize()
        for i in range(0, len(sc), 7 if len(sc) > 8 else 1):
            s = _solver(amd, sc[i])
            one = torch.zeros(steps, 1, device="cuda")
            s.run(acc[i], steps, [lis[i]], one)
            assert torch.equal(one[:, 0], out[:, i])
            assert np.array_equal(s.get_grid(0).view(np.uint32), hs[i].get_grid(0).view(np.uint32))
            s.adjoint_reset(steps - 1)
            g = torch.zeros(steps, s.nt, device="cuda")
            s.adjoint_run(w[:, i].contiguous(), steps, [lis[i]], g)
            torch.cuda.synchronize()
            assert torch.equal(g, grads[i])
