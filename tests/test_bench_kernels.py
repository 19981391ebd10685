"""bench.py finds its kernels' dispatches in a profile by name: the roofline's HBM traffic is read from
counter passes, and a kernel that became a template has its arguments in its name."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.parametrize("name,kernel,same", [
    ("pppm_amd::(anonymous namespace)::k_near(pppm_amd::SceneStep, int, int)", "k_near", True),
    ("void pppm_amd::(anonymous namespace)::k_dirichlet<false>(pppm_amd::SceneStep)", "k_dirichlet", True),
    ("void pppm_amd::(anonymous namespace)::k_dirichlet<(bool)1>(pppm_amd::SceneStep)", "k_dirichlet", True),
    ("void pppm_amd::(anonymous namespace)::k_fdtd_march<true>(float*, pppm_amd::FdtdParams)", "k_fdtd_march", True),
    ("k_dirichlet", "k_dirichlet", True),
    ("k_far.kd", "k_far", True),
    ("void pppm_amd::(anonymous namespace)::k_batch_dirichlet<true>(pppm_amd::SceneStep const*)", "k_dirichlet", False),
    ("pppm_amd::(anonymous namespace)::k_face_far(pppm_amd::SceneStep)", "k_far", False),
    ("pppm_amd::(anonymous namespace)::k_batch_near(pppm_amd::SceneStep const*)", "k_near", False),
    ("__amd_rocclr_copyBuffer", "k_near", False)])
def test_dispatch_names(name, kernel, same):
    import bench
    assert bench.is_kernel(name, kernel) == same

