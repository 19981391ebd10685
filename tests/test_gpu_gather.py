"""The segmented gathers of the step: lists shorter and longer than a round (64 pairs) and a chunk
(256), against the oracle; and one, two or four wave-map entries per wave (chosen by the number of
waves a launch has), against each other. All bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N, H, C = 20, 0.01, 343.0
DT = float(np.float32(H / (np.sqrt(3.0) * C)))


def _cluster(n, seed=0, spread=0.02):
    """n separate small triangles around the grid's centre."""
    rng = np.random.default_rng(seed)
    c = N * H / 2 + rng.uniform(-spread, spread, (n, 1, 3))
    v = (c + rng.uniform(-0.003, 0.003, (n, 3, 3))).reshape(-1, 3)
    return v.astype(np.float32), np.arange(3 * n, dtype=np.int32).reshape(n, 3)


# pairs per cell / per triangle: all lists of one pair; one list of 63, 64, 65, 255, 257 pairs per
# triangle and cell (every triangle in the same cell); 600 triangles over several cells
@pytest.mark.parametrize("n,spread", [(1, 0.02), (2, 0.02), (63, 1e-4), (64, 1e-4), (65, 1e-4), (255, 1e-4),
                                      (257, 1e-4), (600, 0.02)])
def test_list_lengths_against_the_oracle(amd, oracle_mod, n, spread):
    import torch
    v, f = _cluster(n, seed=n, spread=spread)
    g = amd.PPPMSolver(N, H, DT, (0, 0, 0), 0, 0.83, C)
    o = oracle_mod.Oracle(N, H, DT, (0, 0, 0), C, 0.83, oracle_mod.FP64)
    g.set_mesh(v, f)
    o.set_mesh(v, f)
    rng = np.random.default_rng(7)
    # separate triangles in one cell couple strongly: short runs of small inputs stay finite
    steps = 20
    acc = rng.standard_normal((steps, n)).astype(np.float32)
    out = torch.zeros(steps, 2, device="cuda")
    lis = [(N // 2, N // 2, N // 2), (N // 2 + 3, N // 2, N // 2 - 2)]
    g.run(torch.from_numpy(acc).cuda(), steps, lis, out)
    ref = np.zeros((steps, 2), np.float32)
    for i in range(steps):
        o.step(acc[i])
        ref[i] = [o.read(*x) for x in lis]
    assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(g.get_grid(0).view(np.uint32).reshape(-1), o.grid(0).view(np.uint32).reshape(-1))
    for a, b in zip(g.get_history(), o.history()):
        assert np.array_equal(a.view(np.uint32), np.asarray(b).view(np.uint32).reshape(a.shape))


def _gran(waves):
    """Wave-map entries a wave takes in a launch of that many (gather_gran)."""
    return 4 if waves >= 32768 else 2 if waves >= 16384 else 1


# edge, scenes of 5120 triangles, entries per wave of the cell gathers and of the face gather (one scene
# has 2161 cell entries and 4000 to 9000 face entries)
@pytest.mark.parametrize("edge,n_scenes,cells,faces", [(56, 1, 1, 1), (56, 3, 1, 2), (56, 8, 2, 4), (48, 16, 4, 4)])
def test_entries_per_wave_agree(amd, scenes_mod, edge, n_scenes, cells, faces):
    """Scenes together, one, two or four entries a wave, against each scene alone (one entry): samples
    inside and outside the corrected region, grids and histories."""
    import torch
    sc = [scenes_mod.c3_scene(edge, 4, seed=i, steps=6) for i in range(n_scenes)]

    def solvers():
        s = [amd.PPPMSolver(x.res, x.dl, x.dt, x.min_pos, 0, 0.83, x.c) for x in sc]
        for a, x in zip(s, sc):
            a.set_mesh(x.verts, x.tris)
        return s
    rng = np.random.default_rng(1)
    acc = [torch.from_numpy(rng.standard_normal((6, len(x.tris))).astype(np.float32)).cuda() for x in sc]
    together = solvers()
    lis, w3, w4 = [], [], []
    for s in together:
        c3 = s.get_c3()[0]
        q = int(c3[len(c3) // 2])
        lis.append([(q // edge ** 2, q // edge % edge, q % edge), (7 * edge // 8,) * 3])
        assert (lis[-1][1][0] * edge + lis[-1][1][1]) * edge + lis[-1][1][2] not in c3
        # entries by the lists' capacities: 16 face pairs a triangle, or what a first mesh grew to
        p4, room = s.stats()["P4"], 16 * s.nt + 1024
        w3.append(27 * s.nt // 64 + 1)
        w4.append((room if p4 <= room else p4 * 5 // 4 + 1024) // 64 + 1)
    assert (_gran(sum(w3)), _gran(sum(w4))) == (cells, faces), (sum(w3), sum(w4))
    assert all((_gran(a), _gran(b)) == (1, 1) for a, b in zip(w3, w4))
    out = torch.zeros(6, n_scenes, 2, device="cuda")
    amd.PPPMBatch(together).run(acc, 6, lis, out)
    for i, s in enumerate(solvers()):
        one = torch.zeros(6, 2, device="cuda")
        s.run(acc[i], 6, lis[i], one)
        assert torch.equal(one.view(torch.int32), out[:, i].contiguous().view(torch.int32))
        assert one[:, 0].abs().max() > 0
        assert np.array_equal(s.get_grid(0).view(np.uint32), together[i].get_grid(0).view(np.uint32))
        for a, b in zip(s.get_history(), together[i].get_history()):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_step_routes_agree(amd, scenes_mod):
    """The step in three launches, by series (windows handed from step to step) and alone, equals
    the phase entry points and the launches of the timed step, in any order of calls."""
    import torch
    sc = scenes_mod.c1_static_sphere(steps=40)
    rng = np.random.default_rng(2)
    acc = rng.standard_normal((40, len(sc.tris))).astype(np.float32)
    dev = torch.from_numpy(acc).cuda()
    lis = [sc.listener, (16, 16, 23)]

    def solver():
        s = amd.PPPMSolver(sc.res, sc.dl, sc.dt, sc.min_pos, 0, 0.83, sc.c)
        s.set_mesh(sc.verts, sc.tris)
        return s

    def phases(s, i):
        s.fdtd_step()
        s.solve_fdtd_far()
        s.set_neumann_condition(acc[i])
        s.update_dirichlet()
        s.solve_fdtd_near()
    a, b = solver(), solver()
    for i in range(40):
        phases(a, i)
    out = torch.zeros(40, 2, device="cuda")
    b.run(dev[:7], 7, lis, out[:7], use_graph=False)
    b.update_grid_and_face(acc[7])
    phases(b, 8)
    b.run(dev[9:20], 11, lis, out[9:20], use_graph=True)
    b.set_timing(True)
    b.update_grid_and_face(acc[20])
    b.run(dev[21:24], 3, lis, out[21:24], use_graph=False)
    b.set_timing(False)
    b.run_noalloc(dev[24:27], 3, lis, out[24:27])
    b.update_grid_and_face(dev[27])
    b.run(dev[28:], 12, lis, out[28:], use_graph=False)
    assert a.time_idx() == b.time_idx()
    for rel in (0, -1):
        assert np.array_equal(a.get_grid(rel).view(np.uint32), b.get_grid(rel).view(np.uint32))
    for x, y in zip(a.get_history(), b.get_history()):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    assert np.array_equal(out[-1].cpu().numpy(), b.read_cells(lis))


@pytest.mark.parametrize("route", ["step", "run", "graph", "tail", "moving", "batch", "batch_full", "batch_tail"])
def test_phases_behind_a_step(amd, scenes_mod, route):
    """The far field that a step used stays for the phases called after it: another Neumann input, the
    Dirichlet update and the near field again, against steps made of phases. tail: six steps behind two
    graphs of 32 (batch_tail: none). batch_full: scenes enough for a face far field launch of its own."""
    import torch
    full = route == "batch_full"
    steps = {"tail": 70, "batch_tail": 64}.get(route, 6)
    sc = scenes_mod.c3_scene(56, 4, seed=2, steps=6) if full else scenes_mod.c1_static_sphere(steps=6)
    rng = np.random.default_rng(5)
    acc = rng.standard_normal((steps + 2, len(sc.tris))).astype(np.float32)
    dev, lis = torch.from_numpy(acc).cuda(), [sc.listener]
    out = torch.zeros(steps, 1, device="cuda")

    def solver():
        s = amd.PPPMSolver(sc.res, sc.dl, sc.dt, sc.min_pos, 0, 0.83, sc.c)
        s.set_mesh(sc.verts, sc.tris)
        return s
    a, b = solver(), solver()
    if route == "step":
        for i in range(6):
            b.update_grid_and_face(acc[i])
    elif route == "moving":
        rows = torch.from_numpy(np.repeat(sc.verts.reshape(1, -1), 6, 0).astype(np.float32)).cuda()
        b.run_moving(rows, dev, 6, lis, out)
    elif route.startswith("batch"):
        n = 8 if full else 1
        amd.PPPMBatch([b] + [solver() for _ in range(n - 1)]).run([dev] * n, steps, lis * n,
                                                                 torch.zeros(steps, n, device="cuda"))
    else:
        b.run(dev, steps, lis, out, use_graph=route != "run")
    for i in range(steps):
        a.fdtd_step()
        a.solve_fdtd_far()
        a.set_neumann_condition(acc[i])
        a.update_dirichlet()
        a.solve_fdtd_near()
    for i in (steps - 1, steps, steps + 1):  # the step's own input again, then others
        for s in (a, b):
            s.set_neumann_condition(acc[i])
            s.update_dirichlet()
            s.solve_fdtd_near()
        assert np.array_equal(a.get_grid(0).view(np.uint32), b.get_grid(0).view(np.uint32)), i
        for x, y in zip(a.get_history(), b.get_history()):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), i
    assert np.abs(a.get_grid(0)).max() > 0
