"""Latent attention's preparation in 16-byte requests (csrc/latent.hip latent_prep_vec_kernel): more norm columns than a wave's first request, more rotated heads than its
threads, a shared key that is rotated in part, and sizes that stay element by element (test_gpu_mixers.py has the comparison and its tolerances)."""
import pytest
from test_gpu_mixers import TYPES, ops, test_latent_prep as compare  # noqa: F401

pytestmark = pytest.mark.gpu


@TYPES
@pytest.mark.parametrize("H,dn,dr,R,n_rot,ring", [(2, 8, 40, 1032, 16, 9), (70, 16, 64, 64, 64, 5), (1, 0, 16, 8, 16, 3), (2, 8, 16, 520, 8, 9), (3, 4, 16, 64, 16, 9)])
def test_sizes(ops, dt, H, dn, dr, R, n_rot, ring):  # noqa: F811
    compare(ops, dt, H, dn, dr, R, n_rot, ring)
