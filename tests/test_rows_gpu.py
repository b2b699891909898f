"""The weight-streaming kernels for few rows (csrc/rows.hip) at the edges of
their row blocks, K tiles and column blocks, against the oracle."""
import numpy as np
import pytest
import torch

import omni_int8 as oi

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


# Rows at the edges of the row blocks; K of one partial tile, tiles of 128 and
# 256 bytes with and without a partial last one, fewer tiles than waves;
# columns of one partial block, either side of one block per CU (16 x 256),
# and more than 512 per workgroup.
@pytest.mark.parametrize("rows,width,columns", [
    (1, 16, 1), (4, 240, 17), (5, 256, 15), (8, 272, 4096), (9, 2064, 33), (16, 4304, 100),
    (17, 144, 31), (32, 1168, 64), (33, 128, 47), (48, 3072, 130), (49, 112, 16), (64, 4112, 95),
    (3, 512, 4097), (7, 1152, 4112), (16, 400, 5001), (31, 528, 4100), (47, 384, 4129), (64, 656, 4128),
    (2, 64, 140001), (13, 32, 140001), (64, 48, 131104)])
def test_w8a8_stream_bit_exact(oracle, rows, width, columns):
    rng = np.random.default_rng(rows * 7 + width + columns)
    codes = rng.integers(-128, 128, (rows, width), dtype=np.int8)
    w = rng.integers(-128, 128, (columns, width), dtype=np.int8)
    rs = rng.uniform(1e-4, 1e-2, rows).astype(np.float32)
    scale = rng.uniform(0.002, 0.02, columns).astype(np.float32)
    bias = rng.standard_normal(columns).astype(np.float32)
    acc = oracle.int8_acc(codes, w)
    # small and wide (wrapping) sums and zero points, and none
    small = (rng.integers(-5000, 5000, rows).astype(np.int32), rng.integers(-3, 4, columns).astype(np.int32))
    wide = (rng.integers(-2**31, 2**31, rows).astype(np.int32), rng.integers(-2**31, 2**31, columns).astype(np.int32))
    none = (np.zeros(rows, np.int32), np.zeros(columns, np.int32))
    for total, zero in (small, wide, none):
        t, z = (None, None) if total is none[0] else (dev(total), dev(zero))
        got, dump = oi.w8a8_gemm(dev(codes), dev(rs), t, dev(w), dev(scale), z, acc_dump=True)
        o32, _ = oracle.w8a8_finish(acc, total, rs, scale, zero)
        assert np.array_equal(host(dump), acc)
        assert np.array_equal(host(got).view(np.uint32), o32.view(np.uint32))
        got = oi.w8a8_gemm(dev(codes), dev(rs), t, dev(w), dev(scale), z, dev(bias), torch.float16)
        _, o16 = oracle.w8a8_finish(acc, total, rs, scale, zero, bias)
        assert np.array_equal(host(got).view(np.uint16), o16)
