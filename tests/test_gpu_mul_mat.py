"""mtg_q8_mul_mat_dev at the edges of its one-launch kernel (csrc/kernels.hip k_mul_mat):
K below four block pairs (empty K-slices) and at the LDS panel's limit for 8 and 16
rows (beyond it the general path runs), 1,024 and 1,025 tiles (a workgroup or a wave
per tile), unaligned operands. Bit-identical to the oracle."""
import ctypes

import numpy as np
import pytest
import torch

import mtg
import oracle_py

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n,T,shift", [(64, 16, 1, 0), (64, 16, 16, 0), (192, 48, 7, 0), (320, 16 * 1024, 9, 0),
                                         (320, 16 * 1025, 9, 0), (128, 16 * 1025, 3, 0), (14528, 32, 8, 0),
                                         (14592, 32, 8, 0), (7232, 32, 9, 0), (7296, 32, 16, 0), (1024, 64, 2, 1)])
def test_mul_mat_edges(k, n, T, shift):
    print("mul_mat: k %d n %d T %d shift %d" % (k, n, T, shift), flush=True)
    rng = np.random.default_rng(k + n + T)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    raw = np.empty(n * (k // 32) * 34, np.uint8)
    mtg.lib().mtg_quantize_q8_0_weight(mtg.ptr(w), n * k, mtg.ptr(raw))
    x = rng.standard_normal((T, k)).astype(np.float32)
    x[0, :32] = 0.0
    ref = oracle_py.mul_mat(mtg.TYPE_Q8_0, raw, k, n, x)
    packed = ctypes.c_void_p()
    assert mtg.lib().mtg_q8_pack(mtg.ptr(raw), k, n, ctypes.byref(packed)) == 0
    xd = torch.zeros(T * k + 4, device="cuda")
    yd = torch.full((T * n + 8,), 7.0, device="cuda")
    xd[shift:shift + T * k] = torch.from_numpy(x.reshape(-1)).cuda()
    rc = mtg.lib().mtg_q8_mul_mat_dev(packed, ctypes.c_void_p(xd.data_ptr() + 4 * shift), T,
                                      ctypes.c_void_p(yd.data_ptr() + 4 * shift))
    mtg.lib().mtg_q8_free(packed)
    assert rc == 0
    y = yd.cpu().numpy()
    assert np.array_equal(y[shift:shift + T * n].reshape(T, n), ref)
    assert (y[:shift] == 7.0).all() and (y[shift + T * n:] == 7.0).all()


@pytest.mark.parametrize("k,n,T,y_at", [(1024, 1024, 1, 0), (1024, 1024, 16, 0), (256, 256, 8, 255), (256, 256, 9, -255),
                                        (1024, 512, 16, 64)])
def test_mul_mat_over_its_own_input(k, n, T, y_at):
    """y over x, or y_at floats away from its start: x is read before y is written."""
    print("mul_mat over x: k %d n %d T %d y at x %+d" % (k, n, T, y_at), flush=True)
    rng = np.random.default_rng(k + n + T)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    raw = np.empty(n * (k // 32) * 34, np.uint8)
    mtg.lib().mtg_quantize_q8_0_weight(mtg.ptr(w), n * k, mtg.ptr(raw))
    x = rng.standard_normal((T, k)).astype(np.float32)
    ref = oracle_py.mul_mat(mtg.TYPE_Q8_0, raw, k, n, x)
    packed = ctypes.c_void_p()
    assert mtg.lib().mtg_q8_pack(mtg.ptr(raw), k, n, ctypes.byref(packed)) == 0
    buf = torch.full((T * max(k, n) + 512,), 7.0, device="cuda")
    xo, yo = 256, 256 + y_at
    buf[xo:xo + T * k] = torch.from_numpy(x.reshape(-1)).cuda()
    torch.cuda.synchronize()
    rc = mtg.lib().mtg_q8_mul_mat_dev(packed, ctypes.c_void_p(buf.data_ptr() + 4 * xo), T,
                                      ctypes.c_void_p(buf.data_ptr() + 4 * yo))
    mtg.lib().mtg_q8_free(packed)
    assert rc == 0
    got = buf.cpu().numpy()
    assert np.array_equal(got[yo:yo + T * n].reshape(T, n), ref)
    assert (got[:min(xo, yo)] == 7.0).all() and (got[max(xo + T * k, yo + T * n):] == 7.0).all()


@pytest.mark.parametrize("k,n,T", [(4160, 4096, 16), (4160, 4112, 9), (8640, 8192, 1), (8704, 4112, 8), (8704, 8192, 1)])
def test_mul_mat_large_panels(k, n, T):
    """Both sides of the choice by the panels a CU holds (one, two; more tiles than that)."""
    print("mul_mat, large panels: k %d n %d T %d" % (k, n, T), flush=True)
    rng = np.random.default_rng(k + n + T)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    raw = np.empty(n * (k // 32) * 34, np.uint8)
    mtg.lib().mtg_quantize_q8_0_weight(mtg.ptr(w), n * k, mtg.ptr(raw))
    x = rng.standard_normal((T, k)).astype(np.float32)
    packed = ctypes.c_void_p()
    assert mtg.lib().mtg_q8_pack(mtg.ptr(raw), k, n, ctypes.byref(packed)) == 0
    xd, yd = torch.from_numpy(x).cuda(), torch.zeros(T, n, device="cuda")
    rc = mtg.lib().mtg_q8_mul_mat_dev(packed, ctypes.c_void_p(xd.data_ptr()), T, ctypes.c_void_p(yd.data_ptr()))
    mtg.lib().mtg_q8_free(packed)
    assert rc == 0
    assert np.array_equal(yd.cpu().numpy(), oracle_py.mul_mat(mtg.TYPE_Q8_0, raw, k, n, x))
