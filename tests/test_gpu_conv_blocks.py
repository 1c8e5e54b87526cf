"""Convolutions that the pipelined kernel does not take: outputs whose 8-byte
granules are not aligned, with one to four output blocks per workgroup.

Inputs and weights are small whole numbers, so every sum is exact in FP32 and
the BF16 results must equal the oracle's.
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


def _conv(xd, wd, bd, out, off, kc, nc, md, dims):
    from efwi import _native as N
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert N.lib().efwi_nn_conv3(_p(xd), kc, kc, _p(wd), _p(bd), _p(out, off), nc, nc, _p(md), nc, *dims, 0, 1, s) == 0


# 1134 bricks of 64 voxels, 1088 of 32 (four workgroups per CU and more), few bricks
@pytest.mark.parametrize("dims,kc,nc,off", [((33, 125, 66), 16, 48, 4), ((33, 125, 66), 16, 32, 4), ((33, 125, 66), 16, 64, 1),
                                            ((33, 125, 66), 32, 48, 2), ((33, 125, 66), 32, 32, 4), ((33, 63, 50), 16, 64, 4),
                                            ((33, 63, 50), 16, 48, 4), ((33, 63, 50), 32, 64, 4), ((5, 7, 70), 16, 64, 4)])
@pytest.mark.parametrize("masked", [0, 1])
def test_convolution(dims, kc, nc, off, masked):
    rng = np.random.default_rng(sum(dims) + kc + nc)
    V = int(np.prod(dims))
    ints = lambda *n: rng.integers(-2, 3, n).astype(np.float32)  # noqa: E731
    dev = lambda a: torch.from_numpy(a).to(DEV).to(torch.bfloat16)  # noqa: E731
    x, w, b, m = ints(*dims, kc), ints(27, nc, kc), ints(nc), ints(V, nc)
    print(f"[gpu] conv blocks {dims} {kc}->{nc} offset {off} masked {masked}", flush=True)
    out = torch.full(((V + 1) * nc,), 7.0, dtype=torch.bfloat16, device=DEV)
    _conv(dev(x.reshape(V, kc)), dev(w), torch.from_numpy(b).to(DEV), out, off, kc, nc, dev(m) if masked else None, dims)
    ref = np.maximum(O.conv3(x, w).reshape(V, nc) + b, 0)
    if masked:
        ref = np.where(m > 0, ref, 0)
    got = out.float().cpu().numpy()
    np.testing.assert_array_equal(got[off:off + V * nc].reshape(V, nc), O.bf16_round(ref.astype(np.float32)))
    assert np.all(got[:off] == 7.0) and np.all(got[off + V * nc:] == 7.0)


def test_output_blocks_share_the_input():
    """Three unaligned output blocks of one input take less time than three
    convolutions of one block (they load the input once)."""
    dims = (96, 128, 128)
    V = int(np.prod(dims))
    x = torch.randn(V, 16, device=DEV).bfloat16()
    args = {}
    for nc in (16, 48):
        w, b = torch.randn(27, nc, 16, device=DEV).bfloat16(), torch.randn(nc, device=DEV)
        args[nc] = (x, w, b, torch.empty(V * nc + 4, device=DEV, dtype=torch.bfloat16), 4, 16, nc, None, dims)
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    us = {16: [], 48: []}
    for _ in range(8):
        for nc in us:
            _conv(*args[nc])
            e[0].record()
            for _ in range(20):
                _conv(*args[nc])
            e[1].record()
            e[1].synchronize()
            us[nc].append(e[0].elapsed_time(e[1]) / 20 * 1e3)
    best = {nc: min(t) for nc, t in us.items()}
    print(f"[gpu] unaligned 16->16 {best[16]:.1f} us, 16->48 {best[48]:.1f}", flush=True)
    assert best[48] < 3 * best[16]
