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
