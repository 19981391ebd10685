"""reset, save_state and load_state as one launch over word ranges: odd grids and meshes (ranges that
start off 16-byte boundaries), state buffers at every alignment, byte-aligned ones included (those take
copies)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
H, C = 0.01, 343.0
DT = float(np.float32(H / (np.sqrt(3.0) * C)))


def _solver(amd, n, nt):
    rng = np.random.default_rng(nt)
    c = n * H / 2 + rng.uniform(-0.02, 0.02, (nt, 1, 3))
    v = (c + rng.uniform(-0.003, 0.003, (nt, 3, 3))).reshape(-1, 3).astype(np.float32)
    s = amd.PPPMSolver(n, H, DT, (0, 0, 0), 0, 0.83, C)
    s.set_mesh(v, np.arange(3 * nt, dtype=np.int32).reshape(nt, 3))
    return s


def _state(s):
    return [s.get_grid(r).copy() for r in (0, -1)] + [np.array(x) for x in s.get_history()]


@pytest.mark.parametrize("n,nt", [(20, 1), (20, 64), (23, 3), (33, 131)])
@pytest.mark.parametrize("offset", [0, 16, 4, 1])
def test_state_round_trip(amd, n, nt, offset):
    import torch
    a, b = _solver(amd, n, nt), _solver(amd, n, nt)
    acc = torch.from_numpy(np.random.default_rng(0).standard_normal((9, nt)).astype(np.float32)).cuda()
    out, out2 = torch.zeros(4, 1, device="cuda"), torch.zeros(4, 1, device="cuda")
    lis = [(n // 2, n // 2, n // 2)]
    a.run(acc[:5], 5, lis, torch.zeros(5, 1, device="cuda"))
    size = a.state_bytes()
    buf = torch.full((size + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    a.save_state(buf[offset:offset + size])
    got = buf.cpu().numpy()
    assert np.all(got[:offset] == 0xA5) and np.all(got[offset + size:] == 0xA5)
    want = _state(a)
    body = np.concatenate([x.astype(np.float32).ravel() for x in want[:2]]).view(np.uint8)
    assert np.array_equal(got[offset:offset + body.size], body)
    assert tuple(got[offset + size - 16:offset + size].copy().view(np.int32)) == (a.time_idx(), n, nt, 0x5157)
    b.load_state(buf[offset:offset + size])
    assert b.time_idx() == a.time_idx()
    for x, y in zip(_state(b), want):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    a.run(acc[5:], 4, lis, out)
    b.run(acc[5:], 4, lis, out2)
    assert torch.equal(out, out2)
    a.reset()
    assert a.time_idx() == -1 and all(not x.any() for x in _state(a))


@pytest.mark.parametrize("missing", [0, 4, 16, 80, 300])
def test_buffer_too_small_is_refused(amd, missing):
    """A buffer that ends before the state does (by less than its allocation's last page holds) is
    refused through the C ABI, which has only the pointer; one of exactly the state's size is not."""
    import ctypes
    import torch
    torch.cuda.init()
    a = _solver(amd, 20, 3)
    a.run(torch.ones(2, 3, device="cuda"), 2, [(10, 10, 10)], torch.zeros(2, 1, device="cuda"))
    torch.cuda.synchronize()
    size = a.state_bytes()
    assert -size % 4096 >= 16 and missing < size % 4096  # past the buffer is still the same page
    p = ctypes.c_void_p()  # (the library's handle also finds the HIP runtime it is linked to)
    assert a.lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size - missing)) == 0
    try:
        rc = a.lib.pppm_save_state(a.h, p)
        assert (rc != 0) == (missing > 0)
        a.save_state(torch.empty(size, dtype=torch.uint8, device="cuda"))  # the refusal leaves no error behind
        if not missing:
            want = _state(a)
            a.reset()
            assert a.lib.pppm_load_state(a.h, p) == 0 and a.time_idx() == 1
            for x, y in zip(_state(a), want):
                assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
        torch.cuda.synchronize()
    finally:
        assert a.lib.hipFree(p) == 0


def test_save_state_is_captured(amd):
    """save_state in a caller's graph, replayed, with steps of the caller's own between the replays."""
    import torch
    a = _solver(amd, 23, 5)
    side = torch.cuda.Stream()
    a.set_stream(side.cuda_stream)
    size = a.state_bytes()
    buf, want = (torch.zeros(size, dtype=torch.uint8, device="cuda") for _ in range(2))
    acc, out = torch.ones(3, 5, device="cuda"), torch.zeros(3, 1, device="cuda")
    torch.cuda.synchronize()
    a.run(acc, 3, [(11, 11, 11)], out)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        a.save_state(buf)
    for _ in range(3):  # three steps move the levels round to where they were captured
        torch.cuda.synchronize()
        a.run(acc, 3, [(11, 11, 11)], out)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        a.save_state(want)
        torch.cuda.synchronize()
        assert torch.equal(buf[:size - 16], want[:size - 16])  # the time index is the captured one
