"""The weight-streaming kernels for few rows (csrc/rows.hip) at the edges of
their row blocks, K tiles and column blocks, against the oracle."""
import numpy as np
import pytest
import torch

import omni_int8 as oi
import tolerance
from omni_int8 import f16

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
    w8a8_case(oracle, rows, width, columns)


# More than 64 rows in tiles of 48 and 64 by 32 (30) and 64 (31) columns: ragged
# in each direction, partial K tiles, more units than one workgroup per CU
# holds, more than eight units per workgroup.
@pytest.mark.parametrize("tile", ["30", "31"])
@pytest.mark.parametrize("rows,width,columns", [
    (65, 64, 33), (96, 144, 64), (97, 1040, 65), (128, 528, 130), (129, 16, 31), (190, 2048, 100), (256, 272, 515),
    (300, 96, 6000), (1000, 208, 1100), (2049, 48, 8300)])
def test_w8a8_tiles_bit_exact(oracle, rows, width, columns, tile, knobs):
    knobs.set("OMNI_W8A8_TILE", tile)
    w8a8_case(oracle, rows, width, columns)


# The default route of small matrices.
@pytest.mark.parametrize("rows,width,columns", [(65, 4304, 1152), (100, 1536, 1536), (200, 1152, 777)])
def test_w8a8_tiles_by_default(oracle, rows, width, columns):
    w8a8_case(oracle, rows, width, columns)


def w8a8_case(oracle, rows, width, columns):
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


def close(got, want):
    # f32 sums of products exact in f32 (W4A16: of weights rounded to f16, as
    # the reference's own route rounds them), then one rounding to f16
    assert tolerance.rel_err(host(got), want) <= tolerance.FP16_REL_TOL


# Shapes that the streaming kernels take by default (w8a16_rows_take; three and
# four rows of K % 64 != 0 the GEMV): every row block, K % 64 and K % 256 not 0,
# one block and several per workgroup.
@pytest.mark.parametrize("rows,width,columns", [
    (1, 18944, 40), (4, 16400, 33), (3, 4112, 17), (4, 1552, 8195), (5, 16, 7), (6, 1040, 100), (8, 4624, 4100),
    (8, 1168, 4112), (9, 4112, 64), (16, 240, 31), (13, 4096, 4113), (16, 528, 9000), (17, 64, 16), (32, 1104, 50),
    (31, 336, 4130), (33, 272, 40), (48, 1040, 300), (47, 368, 4100), (49, 144, 30), (64, 2064, 70), (63, 400, 4101),
    (24, 32, 131200), (3, 8256, 17), (4, 1600, 8195), (4, 4160, 2100)])
def test_w8a16_stream(rows, width, columns):
    w8a16_case(rows, width, columns)


# More rows, which the GEMMs take: small matrices, ragged and K % 64 != 0.
@pytest.mark.parametrize("rows,width,columns", [
    (65, 1536, 33), (96, 80, 64), (97, 4608, 65), (128, 208, 130), (192, 4304, 100), (256, 64, 515), (300, 48, 2100),
    (130, 1168, 4300), (2049, 16, 900)])
def test_w8a16_above_64_rows(rows, width, columns):
    w8a16_case(rows, width, columns)


def w8a16_case(rows, width, columns):
    rng = np.random.default_rng(rows + 3 * width + columns)
    x = rng.standard_normal((rows, width)).astype(np.float16)
    w = rng.integers(-128, 128, (columns, width), dtype=np.int8)
    scale = rng.uniform(0.002, 0.02, columns).astype(np.float16)
    bias = rng.standard_normal(columns).astype(np.float16)
    exact = (x.astype(np.float64) @ w.T.astype(np.float64)) * scale.astype(np.float64)
    close(oi.w8a16_linear(dev(x), dev(w), dev(scale)), exact)
    close(oi.w8a16_linear(dev(x), dev(w), dev(scale), dev(bias)), exact + bias.astype(np.float64))
    # a row's infinity stays in its row (times a weight of 0 it is NaN), also in
    # the last one, which the kernels' row blocks repeat
    for row in {0, rows - 1}:
        y = x.copy()
        y[row, width - 1] = np.inf
        got = host(oi.w8a16_linear(dev(y), dev(w), dev(scale)))
        assert not np.isfinite(got[row]).any()
        assert np.isfinite(np.delete(got, row, 0)).all()


@pytest.mark.parametrize("rows,width,columns", [
    (1, 33024, 20), (3, 256, 5), (4, 2304, 33), (4, 4352, 2050), (3, 4352, 4100), (4, 512, 4100), (4, 256, 20000),
    (5, 256, 15), (8, 1792, 100), (7, 768, 4100), (9, 3328, 17), (16, 256, 64), (13, 1280, 4097), (17, 512, 31),
    (32, 2816, 70), (29, 768, 4129), (6, 256, 131100), (5, 128, 33), (8, 1152, 100), (16, 2944, 4099), (3, 4224, 2051),
    (32, 1408, 65), (17, 384, 4130), (33, 128, 47), (48, 640, 4100), (40, 1408, 130), (47, 256, 131104),
    (49, 256, 33), (64, 1152, 70), (63, 384, 4099), (3, 256, 1411), (4, 2304, 1409)])
def test_w4a16_stream(oracle, rows, width, columns):
    w4a16_case(rows, width, columns)


def test_w4a16_very_wide():  # the GEMM, whose tiles outnumber the CUs four times
    w4a16_case(56, 128, 131100)


def w4a16_case(rows, width, columns):
    rng = np.random.default_rng(rows + 5 * width + columns)
    x = rng.standard_normal((rows, width)).astype(np.float16)
    packed = rng.integers(0, 256, (columns, width // 2), dtype=np.uint8)
    scale = torch.from_numpy(rng.uniform(0.002, 0.02, (columns, width // 128)).astype(np.float32)).bfloat16()
    bias = rng.standard_normal(columns).astype(np.float16)
    q = np.stack((packed & 15, packed >> 4), -1).reshape(columns, width).astype(np.float64) - 8
    exact = x.astype(np.float64) @ (q * np.repeat(scale.double().numpy(), 128, 1)).T
    close(oi.w4a16_linear(dev(x), dev(packed), scale.cuda()), exact)
    close(oi.w4a16_linear(dev(x), dev(packed), scale.cuda(), dev(bias)), exact + bias.astype(np.float64))


# Group scales outside f16's normal range enter in f32: the result is off by its
# rounding to f16 (half a unit, 2^-11 of the value or 2^-25) and by the f32 sums'
# (2^-24 of the absolute sum for each of `width` additions), no more.
@pytest.mark.parametrize("low,high", [(1e-6, 5e-5), (8192.0, 65536.0)])
@pytest.mark.parametrize("rows,width,columns", [
    (3, 256, 2100), (4, 640, 33), (8, 384, 100), (16, 512, 4200), (32, 128, 70),
    (48, 384, 40), (64, 256, 4100), (4, 640, 1411)])
def test_w4a16_stream_scales(rows, width, columns, low, high):
    rng = np.random.default_rng(rows + width + columns)
    x = (rng.standard_normal((rows, width)) * (1.0 if high < 1 else 2e-3)).astype(np.float16)
    packed = rng.integers(0, 256, (columns, width // 2), dtype=np.uint8)
    scale = torch.from_numpy(rng.uniform(low, high, (columns, width // 128)).astype(np.float32)).bfloat16()
    q = np.stack((packed & 15, packed >> 4), -1).reshape(columns, width).astype(np.float64) - 8
    w = q * np.repeat(scale.double().numpy(), 128, 1)
    exact, total = x.astype(np.float64) @ w.T, np.abs(x.astype(np.float64)) @ np.abs(w).T
    got = host(oi.w4a16_linear(dev(x), dev(packed), scale.cuda())).astype(np.float64)
    bound = np.abs(exact) * 2.0**-11 + 2.0**-25 + width * 2.0**-24 * total
    fits = np.abs(exact) < 65504 * (1 - 2.0**-10)
    assert fits.any() and (np.abs(got - exact) <= bound)[fits].all()


# Where the routes part. Route 1 pins the GEMV (up to 4 rows) or the skinny
# kernel, 2 the GEMM; the streaming kernel's sums, in another order than either's,
# differ in some output's last bit (0).
@pytest.mark.parametrize("rows,width,columns,route", [
    (5, 1024, 4096, 1), (5, 1024, 4112, 1), (8, 1024, 8192, 1), (8, 1024, 8208, 0), (16, 1024, 4352, 1),
    (16, 1024, 4368, 0), (7, 2048, 8176, 1), (7, 2048, 8192, 0), (8, 2048, 4112, 0), (5, 3072, 4112, 0),
    (5, 1040, 4096, 0),
    (3, 7808, 1408, 1), (4, 8192, 2048, 1), (4, 8192, 2064, 0), (4, 8256, 2048, 0), (4, 8272, 2048, 1),
    (4, 4064, 12736, 1), (4, 4160, 12736, 0), (4, 16400, 3000, 0),
    (30, 13760, 9200, 2), (30, 13760, 8192, 0), (30, 13760, 10768, 0), (25, 11904, 9152, 2), (24, 11904, 9152, 0),
    (25, 8192, 9152, 0), (25, 11904, 10752, 2), (31, 5312, 8252, 2), (31, 5184, 8252, 0), (20, 8000, 9728, 2),
    (20, 7872, 9728, 0), (30, 14064, 8576, 0), (36, 1984, 16960, 2), (36, 1920, 16384, 0),
    (50, 1088, 18240, 2), (50, 1088, 14656, 0)])
def test_w8a16_routes(rows, width, columns, route, knobs):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the columns are those of 256 CUs")
    g = torch.Generator(device="cuda").manual_seed(rows + width + columns)
    x = torch.randn((rows, width), generator=g, device="cuda").half()
    w = torch.randint(-127, 128, (columns, width), generator=g, device="cuda", dtype=torch.int8)
    scale = torch.rand(columns, generator=g, device="cuda").half()
    routes_agree(lambda: oi.w8a16_linear(x, w, scale), route, knobs)


@pytest.mark.parametrize("rows,width,columns,route", [
    (4, 7040, 9216, 1), (4, 7168, 9216, 0), (4, 7040, 8192, 0), (4, 7040, 11280, 0), (3, 2432, 1392, 1),
    (3, 2432, 1408, 0), (4, 4352, 2048, 1), (4, 4352, 2064, 0),
    (9, 1152, 8488, 1), (8, 1152, 8488, 0), (24, 1152, 4096, 1), (25, 1152, 4096, 0), (17, 1152, 4112, 0),
    (17, 1280, 2048, 0), (12, 2176, 2200, 1), (13, 2176, 2200, 0), (9, 2304, 2200, 0), (9, 3456, 4096, 1),
    (9, 3712, 4096, 0),
    (61, 5632, 4416, 2), (61, 4096, 4416, 0), (56, 1024, 12288, 2), (56, 1024, 10240, 0), (48, 1024, 12288, 0)])
def test_w4a16_routes(rows, width, columns, route, knobs):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the columns are those of 256 CUs")
    g = torch.Generator(device="cuda").manual_seed(rows + width + columns)
    x = torch.randn((rows, width), generator=g, device="cuda").half()
    w = torch.randint(0, 256, (columns, width // 2), generator=g, device="cuda", dtype=torch.uint8)
    scale = torch.rand((columns, width // 128), generator=g, device="cuda").bfloat16()
    routes_agree(lambda: oi.w4a16_linear(x, w, scale), route, knobs)


def routes_agree(call, route, knobs):
    got = call()
    for pin in ("1", "2"):
        knobs.set("OMNI_W8A16_ROUTE", pin)
        if route in (0, int(pin)):
            assert torch.equal(got, call()) == (route != 0), pin


# A knob at its automatic value leaves the choice as it is without the knob; a
# pin keeps the call off the streaming kernels. The skinny kernel that then
# takes this shape splits K and writes its workspace, they use none.
@pytest.mark.parametrize("name,value,pins", [
    ("ROUTE", 0, False), ("GEMV", 0, False), ("SKINNY", 0, False), ("TILE", 0, False), ("SPLITS", 0, False),
    ("SPLITS", 1, False), ("SKINNY_SPLIT", -1, False), ("ROUTE", 1, True), ("SKINNY", 1, True), ("SPLITS", 2, True),
    ("SKINNY_SPLIT", 4, True)])
def test_automatic_knob_values_pin_nothing(name, value, pins, knobs):
    from omni_int8 import _lib
    L = _lib.lib()
    rows, width, columns = 16, 4096, 14336
    x = torch.randn((rows, width), device="cuda").half()
    out = torch.empty((rows, columns), dtype=torch.float16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for int4 in (False, True):
        if int4 and name == "SKINNY":  # W8A16's alone
            continue
        knobs.set(("OMNI_W4A16_" if int4 and name != "ROUTE" else "OMNI_W8A16_") + name, value)
        ws = torch.full((4 * rows * columns * 4,), 0x5A, dtype=torch.uint8, device="cuda")
        if int4:
            w = torch.randint(0, 256, (columns, width // 2), dtype=torch.uint8, device="cuda")
            scale = torch.rand((columns, width // 128), device="cuda").bfloat16()
            st = L.omni_w4a16_gemm_ws(x.data_ptr(), w.data_ptr(), scale.data_ptr(), 128, None, rows, columns, width,
                                      out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
        else:
            w = torch.randint(-127, 128, (columns, width), dtype=torch.int8, device="cuda")
            scale = torch.rand(columns, device="cuda").half()
            st = L.omni_w8a16_gemm_ws(x.data_ptr(), w.data_ptr(), scale.data_ptr(), None, rows, columns, width,
                                      out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
        assert st == 0, _lib.last_error()
        assert bool((ws != 0x5A).any()) == pins, int4


@pytest.mark.parametrize("rows,width,columns", [
    (5, 32, 9), (8, 160, 100), (9, 1056, 33), (16, 8192, 17), (17, 96, 64), (32, 544, 40), (33, 64, 31),
    (48, 1120, 70), (49, 32, 16), (64, 2080, 95)])
def test_f16_stream(rows, width, columns):
    rng = np.random.default_rng(rows + width + columns)
    x = rng.standard_normal((rows, width)).astype(np.float16)
    w = (rng.standard_normal((columns, width)) * 0.05).astype(np.float16)
    close(f16.depth_try_linear(dev(x), dev(w).t()), x.astype(np.float64) @ w.T.astype(np.float64))


# The 192 x 256 ring: both sides of a tile's edge in rows and columns, one and
# several K tiles per split, whole and split three ways.
@pytest.mark.parametrize("splits", ["1", "3"])
@pytest.mark.parametrize("rows,width,columns", [
    (1, 128, 255), (191, 384, 257), (192, 512, 256), (193, 1408, 300), (385, 640, 770), (500, 2944, 513)])
def test_ring_192(rows, width, columns, splits, knobs):
    for name in ("OMNI_W8A16", "OMNI_W4A16"):
        knobs.set(name + "_TILE", "22")
        knobs.set(name + "_SPLITS", splits)
    rng = np.random.default_rng(rows + width + columns)
    x = rng.standard_normal((rows, width)).astype(np.float16)
    w = rng.integers(-128, 128, (columns, width), dtype=np.int8)
    scale = rng.uniform(0.002, 0.02, columns).astype(np.float16)
    exact = (x.astype(np.float64) @ w.T.astype(np.float64)) * scale.astype(np.float64)
    close(oi.w8a16_linear(dev(x), dev(w), dev(scale)), exact)
    packed = w.view(np.uint8)[:, :width // 2]
    gscale = torch.from_numpy(rng.uniform(0.002, 0.02, (columns, width // 128)).astype(np.float32)).bfloat16()
    q = np.stack((packed & 15, packed >> 4), -1).reshape(columns, width).astype(np.float64) - 8
    exact = x.astype(np.float64) @ (q * np.repeat(gscale.double().numpy(), 128, 1)).T
    close(oi.w4a16_linear(dev(x), dev(packed), gscale.cuda()), exact)
