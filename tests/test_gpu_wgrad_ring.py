"""The weight gradient's brick walk on the GPU: columns along x that end inside
a block's run (and again at the end of a z layer and of a y tile), rows shorter
and longer than a y tile, the smallest volumes, strided operands, and chunk
counts that are no multiple of the XCDs.

The operands are small whole numbers, so every product and sum is exact in FP32
(all partial sums stay below 2^24) in whatever order it is formed: the results
must equal the oracle's.
"""
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
import nn_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _p(t):
    import ctypes as C
    return C.c_void_p(t.data_ptr())


def _dev(a, ld):
    t = torch.full((a.shape[0], ld), 3.0, dtype=torch.bfloat16, device=DEV)
    t[:, :a.shape[1]] = torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(DEV).to(torch.bfloat16)
    return t


# dims, mc, kc, bricks per block, padding of the row strides
CASES = [((1, 1, 1), 16, 16, 1, 0), ((1, 2, 31), 16, 16, 2, 0), ((2, 3, 32), 16, 32, 1, 16),
         ((3, 1, 33), 32, 16, 1, 0), ((5, 7, 33), 16, 16, 3, 16), ((4, 5, 64), 16, 48, 5, 0),
         ((3, 9, 65), 32, 32, 4, 0), ((6, 3, 130), 16, 16, 7, 0), ((5, 4, 40), 48, 16, 100, 0),
         ((9, 11, 5), 16, 16, 1, 0)]


@pytest.mark.parametrize("dims,mc,kc,per,pad", CASES)
def test_brick_walk(dims, mc, kc, per, pad):
    from efwi import _native as N
    import ctypes as C
    rng = np.random.default_rng(sum(dims) + mc + kc)
    V = int(np.prod(dims))
    g = rng.integers(-3, 4, (*dims, mc)).astype(np.float32)
    x = rng.integers(-3, 4, (*dims, kc)).astype(np.float32)
    print(f"[gpu] wgrad walk {dims} {mc}x{kc} per {per}", flush=True)
    gd, xd = _dev(g.reshape(V, mc), mc + pad), _dev(x.reshape(V, kc), kc + pad)
    need = int(N.lib().efwi_nn_wgrad_scratch(mc, kc, *dims, per))
    scr = torch.empty(need, device=DEV)
    dw = torch.full((27, mc, kc), 5.0, device=DEV)
    db = torch.full((mc,), 5.0, device=DEV)
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert N.lib().efwi_nn_wgrad(_p(gd), mc + pad, mc, _p(xd), kc + pad, kc, _p(scr), need, _p(dw), _p(db), *dims, per,
                                 s) == 0
    np.testing.assert_array_equal(dw.cpu().numpy(), O.conv3_wgrad(g, x))
    np.testing.assert_array_equal(db.cpu().numpy(), g.reshape(V, mc).sum(axis=0))


@pytest.mark.parametrize("dims,per", [((2, 2, 2), 1), ((4, 6, 34), 2), ((2, 4, 66), 3), ((6, 2, 64), 4)])
def test_brick_walk_of_an_upsampled_input(dims, per):
    """The same with the input kept as a coarse tensor (read through its
    nearest upsampling) and a second tensor."""
    from efwi import _native as N
    import ctypes as C
    rng = np.random.default_rng(sum(dims))
    mc, k1, k2, V = 16, 32, 16, int(np.prod(dims))
    half = tuple(d // 2 for d in dims)
    g = rng.integers(-3, 4, (*dims, mc)).astype(np.float32)
    c = rng.integers(-3, 4, (*half, k1)).astype(np.float32)
    x2 = rng.integers(-3, 4, (*dims, k2)).astype(np.float32)
    print(f"[gpu] wgrad walk up {dims} per {per}", flush=True)
    gd, cd, xd = _dev(g.reshape(V, mc), mc), _dev(c.reshape(-1, k1), k1), _dev(x2.reshape(V, k2), k2)
    need = int(N.lib().efwi_nn_wgrad_scratch(mc, k1 + k2, *dims, per))
    scr = torch.empty(need, device=DEV)
    dw = torch.full((27, mc, k1 + k2), 5.0, device=DEV)
    db = torch.full((mc,), 5.0, device=DEV)
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert N.lib().efwi_nn_wgrad_cat(_p(gd), mc, mc, _p(cd), k1, k1, 1, _p(xd), k2, k2, _p(scr), need, _p(dw), _p(db),
                                     *dims, per, s) == 0
    ref = O.conv3_wgrad(g, np.concatenate([O.up2(c), x2], axis=3))
    np.testing.assert_array_equal(dw.cpu().numpy(), ref)
    np.testing.assert_array_equal(db.cpu().numpy(), g.reshape(V, mc).sum(axis=0))
