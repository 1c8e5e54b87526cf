"""The pipelined convolution on the GPU at the edges of its range: rows of 32 to
130 voxels, the smallest volumes, partial bricks in every direction, numbers of
bricks around the ones where the output blocks per workgroup change, one to three output
blocks per workgroup, one and several chunks of input channels, inputs kept as
a coarse and a fine tensor, outputs split over two tensors, masks, strided and
unaligned rows.

Inputs and weights are small whole numbers, so every sum is exact in FP32 in
whatever order it is formed, and the BF16 results must equal the oracle's.
"""
import ctypes as C
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
import nn_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _p(t, off=0):
    return None if t is None else C.c_void_p(t.data_ptr() + off * t.element_size())


def _ints(rng, *shape):
    return rng.integers(-2, 3, shape).astype(np.float32)


def _dev(a, ld):
    t = torch.full((a.shape[0], ld), 3.0, dtype=torch.bfloat16, device=DEV)
    t[:, :a.shape[1]] = torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(DEV).to(torch.bfloat16)
    return t


def _host(t):
    return t.float().cpu().numpy()


# dims, input channels, output channels, relu, padding of the row strides, output offset
# (4 channels: 8-byte granules are not aligned)
PLAIN = [((33, 125, 66), 16, 16, 1, 0, 0), ((31, 129, 64), 16, 32, 0, 16, 0), ((33, 63, 127), 16, 48, 1, 0, 0),
         ((29, 131, 65), 32, 32, 0, 0, 0), ((30, 66, 130), 48, 16, 1, 16, 0), ((33, 125, 66), 16, 16, 1, 16, 4),
         # as many workgroups of one output block as CUs, and more
         ((4, 256, 64), 32, 32, 1, 0, 0), ((4, 258, 64), 32, 32, 1, 0, 0), ((16, 32, 32), 64, 64, 0, 0, 0),
         ((24, 32, 32), 64, 64, 1, 16, 0), ((23, 33, 50), 16, 48, 1, 0, 0), ((15, 31, 40), 16, 48, 0, 0, 0),
         ((41, 51, 33), 16, 16, 1, 0, 0),
         # small volumes and short rows
         ((1, 1, 32), 32, 16, 0, 0, 0), ((1, 2, 64), 16, 16, 1, 0, 0), ((5, 7, 33), 48, 16, 1, 16, 0),
         ((9, 6, 63), 32, 32, 0, 0, 0), ((5, 3, 95), 16, 32, 1, 0, 0), ((9, 6, 47), 32, 16, 1, 0, 4)]


@pytest.mark.parametrize("dims,kc,nc,relu,pad,off", PLAIN)
@pytest.mark.parametrize("masked", [0, 1])
def test_convolution(dims, kc, nc, relu, pad, off, masked):
    from efwi import _native as N
    rng = np.random.default_rng(sum(dims) + kc + nc)
    V = int(np.prod(dims))
    x, w, b = _ints(rng, *dims, kc), _ints(rng, 27, nc, kc), _ints(rng, nc)
    print(f"[gpu] conv pipe {dims} {kc}->{nc} masked {masked}", flush=True)
    xd, wd = _dev(x.reshape(V, kc), kc + pad), torch.from_numpy(w).to(DEV).to(torch.bfloat16)
    bd = torch.from_numpy(b).to(DEV)
    out = torch.full((V + 1, nc + pad), 7.0, dtype=torch.bfloat16, device=DEV)
    m = _ints(rng, V, nc) if masked else None
    md = _dev(m, nc) if masked else None
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert N.lib().efwi_nn_conv3(_p(xd), kc + pad, kc, _p(wd), _p(bd), _p(out, off), nc + pad, nc, _p(md), nc, *dims, 0,
                                 relu, s) == 0
    ref = O.conv3(x, w).reshape(V, nc) + b
    if relu:
        ref = np.maximum(ref, 0)
    if masked:
        ref = np.where(m > 0, ref, 0)
    got = _host(out).reshape(-1)[off:off + V * (nc + pad)].reshape(V, nc + pad)
    np.testing.assert_array_equal(got[:, :nc], O.bf16_round(ref.astype(np.float32)))
    # nothing beyond the rows' channels is written
    assert np.all(got[:, nc:] == 7.0) and np.all(_host(out).reshape(-1)[:off] == 7.0)


@pytest.mark.parametrize("dims,k1,k2,n1,n2,up", [((34, 126, 66), 32, 16, 16, 0, 1), ((36, 62, 130), 64, 32, 32, 0, 1),
                                                 ((33, 63, 129), 16, 0, 32, 16, 0), ((33, 65, 127), 32, 0, 64, 32, 0),
                                                 ((31, 129, 65), 16, 32, 16, 0, 0), ((12, 22, 34), 64, 32, 32, 0, 1),
                                                 ((2, 2, 62), 16, 16, 16, 0, 1), ((25, 33, 35), 64, 0, 64, 32, 0)])
def test_joined_inputs_and_outputs(dims, k1, k2, n1, n2, up):
    from efwi import _native as N
    rng = np.random.default_rng(sum(dims) + k1)
    V = int(np.prod(dims))
    d1 = tuple(d // 2 for d in dims) if up else dims
    x1, w = _ints(rng, *d1, k1), _ints(rng, 27, n1 + n2, k1 + k2)
    x2 = _ints(rng, *dims, k2) if k2 else None
    print(f"[gpu] conv pipe cat {dims} {k1}+{k2}->{n1}+{n2} up {up}", flush=True)
    x1d, wd = _dev(x1.reshape(-1, k1), k1), torch.from_numpy(w).to(DEV).to(torch.bfloat16)
    x2d = _dev(x2.reshape(V, k2), k2) if k2 else None
    o1 = torch.full((V, n1), 7.0, dtype=torch.bfloat16, device=DEV)
    o2 = torch.full((V, n2), 7.0, dtype=torch.bfloat16, device=DEV) if n2 else None
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert N.lib().efwi_nn_conv3_cat(_p(x1d), k1, k1, up, _p(x2d), k2, k2, _p(wd), None, _p(o1), n1, n1, _p(o2), n2, n2,
                                     None, 0, *dims, 0, 0, s) == 0
    full = O.up2(x1) if up else x1
    if k2:
        full = np.concatenate([full, x2], axis=3)
    ref = O.bf16_round(O.conv3(full, w).reshape(V, n1 + n2).astype(np.float32))
    np.testing.assert_array_equal(_host(o1), ref[:, :n1])
    if n2:
        np.testing.assert_array_equal(_host(o2), ref[:, n1:])
