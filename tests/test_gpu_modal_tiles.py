"""Modal accelerations at the edges of their tiles (128 triangles by 64 or 128 samples, sixteen
modes at a time, windows of 32 samples) against the oracle, bit for bit, with forces down to where the
products are subnormal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1e3, 1e-37])
@pytest.mark.parametrize("nt,modes,samples", [(1, 1, 1), (63, 7, 31), (64, 8, 32), (65, 9, 33), (130, 65, 64),
                                              (127, 64, 65), (300, 130, 400), (8200, 17, 1029), (8192, 16, 1024), (129, 31, 129)])
def test_tiles_bitexact(amd, oracle_mod, nt, modes, samples, scale):
    import torch
    rng = np.random.default_rng(nt + modes)
    nv = max(nt // 2, 3)
    tris = rng.integers(0, nv, (nt, 3)).astype(np.int32)
    n = rng.standard_normal((nt, 3))
    n = (n / np.linalg.norm(n, axis=1, keepdims=True)).astype(np.float32)
    eig = (rng.standard_normal((3 * nv, modes)) * 0.1).astype(np.float32)
    eigvals = ((2 * np.pi * np.sort(rng.uniform(150.0, 9000.0, modes))) ** 2).astype(np.float32)
    rate = 44100.0
    dt = float(np.float32(1.0) / np.float32(rate))
    ms = amd.ModalSource(eig, eigvals, tris, n, 30.0, 1e-6, rate)
    c = oracle_mod.modal_coeffs(eigvals, dt, 30.0, 1e-6)
    m = oracle_mod.modal_surface_matrix(eig, tris, n)
    state = np.zeros((modes, 3), np.float32)
    accs = torch.full((samples, nt), 7.0, device="cuda")
    for _ in range(2):
        forces = (rng.standard_normal((samples, modes)) * scale).astype(np.float32)
        ms.run(torch.from_numpy(forces).cuda(), accs)
        ref = oracle_mod.modal_accs(m, oracle_mod.modal_iir(c, dt, state, forces))
        assert np.array_equal(accs.cpu().numpy().view(np.uint32), ref.view(np.uint32))
        assert np.array_equal(ms.state().view(np.uint32), state.view(np.uint32))


def test_infinities_and_nan_stay_in_their_sample(amd, oracle_mod):
    """Each accumulator of the matrix cores takes one product at a time: an infinite or NaN force
    spoils the samples that its mode reaches, as the oracle's sums, and no padded or other entry; an
    infinite entry of the surface matrix spoils its triangle alone."""
    import torch
    rng = np.random.default_rng(4)
    nt, modes, samples, nv = 200, 21, 150, 90
    tris = rng.integers(0, nv - 2, (nt, 3)).astype(np.int32)
    tris[77] = (nv - 2, nv - 1, nv - 1)
    n = rng.standard_normal((nt, 3)).astype(np.float32)
    eig = (rng.standard_normal((3 * nv, modes)) * 0.1).astype(np.float32)
    eig[3 * (nv - 1), 20] = np.inf
    eigvals = ((2 * np.pi * np.sort(rng.uniform(150.0, 9000.0, modes))) ** 2).astype(np.float32)
    dt = float(np.float32(1.0) / np.float32(44100.0))
    c = oracle_mod.modal_coeffs(eigvals, dt, 30.0, 1e-6)
    m = oracle_mod.modal_surface_matrix(eig, tris, n)
    assert np.isfinite(np.delete(m, 77, 0)).all() and not np.isfinite(m[77]).all()
    for value, at, mode in [(np.inf, 130, 0), (-np.inf, 149, 16), (np.nan, 140, 20)]:
        ms = amd.ModalSource(eig, eigvals, tris, n, 30.0, 1e-6, 44100.0)
        state = np.zeros((modes, 3), np.float32)
        forces = rng.standard_normal((samples, modes)).astype(np.float32)
        forces[at, mode] = value
        accs = torch.full((samples, nt), 7.0, device="cuda")
        ms.run(torch.from_numpy(forces).cuda(), accs)
        got = accs.cpu().numpy()
        with np.errstate(all="ignore"):
            ref = oracle_mod.modal_accs(m, oracle_mod.modal_iir(c, dt, state, forces))
        assert np.isfinite(np.delete(ref[:at], 77, 1)).all() and not np.isfinite(ref[at]).any()
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        ok = ~np.isnan(ref)
        assert np.array_equal(got[ok].view(np.uint32), ref[ok].view(np.uint32))
