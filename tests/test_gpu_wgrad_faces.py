"""Infinities at the z and x faces of the volume in the weight gradient: a tap's
sum holds the voxel pairs inside the volume only, so an infinite value reaches
the taps that touch its voxel and no other.

Operands are small positive whole numbers (all sums exact in FP32) with one
infinity, so every entry must equal the tap's sum over the overlapping part of
the two tensors, infinite or not.
"""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _p(t):
    return C.c_void_p(t.data_ptr())


def _reference(g, x):
    """dw[t][m][n] = sum_v g[v][m] x[v + d_t][n] over the voxels v with v + d_t inside."""
    out = np.empty((27, g.shape[3], x.shape[3]))
    cut = lambda d, n: (slice(max(0, -d), n - max(0, d)), slice(max(0, d), n - max(0, -d)))  # noqa: E731
    for t in range(27):
        (a, b), (c, d), (e, f) = (cut(k, n) for k, n in zip((t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1), g.shape))
        out[t] = np.einsum("zxym,zxyn->mn", g[a, c, e].astype(np.float64), x[b, d, f].astype(np.float64))
    return out


# even and odd, in one block and over several, rows of a 32- and of a 64-voxel tile
@pytest.mark.parametrize("dims,per", [((4, 4, 64), 2), ((5, 4, 40), 3), ((4, 7, 32), 1), ((3, 3, 70), 20)])
@pytest.mark.parametrize("which", ["src", "dpre"])
def test_infinity_at_a_face(dims, per, which):
    from efwi import _native as N
    rng = np.random.default_rng(sum(dims))
    nz, nx, ny = dims
    V = nz * nx * ny
    for z, x in ((0, 1), (nz - 1, 1), (1, 0), (1, nx - 1), (0, nx - 1), (1, 1)):
        g, a = (rng.integers(1, 4, (*dims, 16)).astype(np.float32) for _ in range(2))
        (a if which == "src" else g)[z, x, 10, 3] = np.inf
        print(f"[gpu] wgrad {dims} per {per}: infinite {which} at ({z}, {x}, 10)", flush=True)
        gd, ad = (torch.from_numpy(t.reshape(V, 16)).to(DEV).to(torch.bfloat16) for t in (g, a))
        need = int(N.lib().efwi_nn_wgrad_scratch(16, 16, *dims, per))
        scr, dw, db = torch.empty(need, device=DEV), torch.empty(27, 16, 16, device=DEV), torch.empty(16, device=DEV)
        s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert N.lib().efwi_nn_wgrad(_p(gd), 16, 16, _p(ad), 16, 16, _p(scr), need, _p(dw), _p(db), *dims, per, s) == 0
        np.testing.assert_array_equal(dw.cpu().numpy(), _reference(g, a))
        np.testing.assert_array_equal(db.cpu().numpy(), g.reshape(V, 16).sum(axis=0))
