"""The batched GEMVs on the f32 matrix core (csrc/dsv4_batch_mf.hip) keep the
single-token GEMV's bits for every (row, token), at the sizes where a plan can
go wrong: row and token tiles of 16 with remainders, rows of one to 256 slots,
a last chunk group inside and across the row's end, tiles split over several
workgroups (the joined forms), scale blocks narrower than a chunk group, and
scale bytes that do not start on a dword. No tolerance: the arithmetic is the
single-token call's, which the other tests hold against the oracle."""
import ctypes

import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu

_KEEP = []          # resident matrices are keyed by host address


def _same(a, b):
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and common.bits_equal(a[~nan], b[~nan])


def _x(rng, nt, cols):
    x = rng.standard_normal((nt, cols), dtype=np.float32)
    x[0, ::3] = -0.0
    x[nt // 2] = (rng.standard_normal(cols) * 1e-39).astype(np.float32)   # subnormal
    x[nt - 1, cols // 2] = np.inf
    return x


def _check(dsv4, m, x, what):
    yn = dsv4.mmq_n(m, x)
    for t in range(x.shape[0]):
        assert _same(yn[t], dsv4.mmq(m, x[t])), (what, t)


# 16384, 12288, 8192 columns: 256, 192, 128 slots, split over 4, 3, 2 or more
# workgroups while the tiles are few; 4112 and 80: a ragged last chunk group;
# 3000 x 7168 and 8200 x 1024: too many tiles to split
@pytest.mark.parametrize("scales", ["e8m0", "f32"])
@pytest.mark.parametrize("rows,cols,nt", [
    (1, 64, 5), (17, 80, 6), (15, 256, 17), (16, 1024, 16), (33, 4112, 33), (300, 4096, 5),
    (1100, 4096, 16), (70, 7168, 64), (2100, 7168, 7), (3000, 7168, 33), (40, 12288, 9),
    (31, 16384, 5), (1030, 16384, 16), (8200, 1024, 20), (129, 8208, 8)])
def test_fp8(gpu, dsv4, rows, cols, nt, scales):
    rng = np.random.default_rng(rows + cols + nt)
    W = common.fp8_codes(rng, (rows, cols))
    Sf, Se = common.fp8_scales(rng, rows, cols)
    S = Se if scales == "e8m0" else Sf
    _KEEP.append((W, S))
    m = dsv4.qmat(W, S)
    up = gpu.dsv4_gpu_upload if scales == "e8m0" else gpu.dsv4_gpu_upload_f32s
    assert up(ctypes.byref(m)) == 0
    _check(dsv4, m, _x(rng, nt, cols), ("fp8", rows, cols, nt, scales))


# rows of 192 slots: split over 3 workgroups below and above one tile per CU
# (4200 rows; 1360 at 33 tokens by the grid's eight row tiles per XCD), 12 waves
# a tile, 6 (8208: a ragged last group), 3, and the least tokens of few rows
@pytest.mark.parametrize("scales", ["e8m0", "f32"])
@pytest.mark.parametrize("rows,cols,nt", [
    (250, 9216, 11), (250, 9216, 12), (500, 10240, 9), (1360, 12288, 33), (4200, 8224, 16),
    (3000, 9216, 48),
    (2200, 8208, 64), (4100, 9216, 64), (4100, 8208, 64)])
def test_fp8_192_slots(gpu, dsv4, rows, cols, nt, scales):
    test_fp8(gpu, dsv4, rows, cols, nt, scales)


@pytest.mark.parametrize("blk_r,blk_c", [(16, 16), (16, 48), (32, 64), (128, 4096)])
def test_fp8_blockings(gpu, dsv4, blk_r, blk_c):
    rows, cols, nt = 75, 2064, 18
    rng = np.random.default_rng(blk_r + blk_c)
    W = common.fp8_codes(rng, (rows, cols))
    S = (127 + rng.integers(-8, -3, size=(-(-rows // blk_r), -(-cols // blk_c)))).astype(np.uint8)
    _KEEP.append((W, S))
    m = dsv4.qmat(W, S, blk_r=blk_r, blk_c=blk_c)
    assert gpu.dsv4_gpu_upload(ctypes.byref(m)) == 0
    _check(dsv4, m, _x(rng, nt, cols), ("fp8", blk_r, blk_c))


@pytest.mark.parametrize("rows,cols,nt", [
    (1, 32, 9), (17, 40, 9), (16, 512, 16), (31, 1048, 20), (300, 4096, 48), (1030, 4096, 64),
    (9000, 1024, 33), (40, 7168, 33), (33, 8200, 10), (20, 12296, 9), (20, 12296, 12),
    (18, 16384, 17)])
def test_bf16(gpu, dsv4, rows, cols, nt):
    rng = np.random.default_rng(rows + cols + nt)
    W = common.bf16_matrix(rng, (rows, cols), 0.02)
    W[0, 0] = 0x7F80                                       # an infinite weight
    _KEEP.append(W)
    m = dsv4.qmat(W, None, wdt=dsv4.WBF16, blk_r=0, blk_c=0)
    assert gpu.dsv4_gpu_upload(ctypes.byref(m)) == 0
    _check(dsv4, m, _x(rng, nt, cols), ("bf16", rows, cols, nt))


@pytest.mark.parametrize("blk_r,blk_c", [(1, 32), (4, 64), (128, 128)])
@pytest.mark.parametrize("rows,cols,nt", [
    (1, 32, 8), (17, 96, 9), (16, 2048, 16), (300, 7168, 24), (1500, 2080, 17), (5000, 1024, 20),
    (33, 8192, 33), (18, 16384, 7)])
def test_fp4(gpu, dsv4, rows, cols, nt, blk_r, blk_c):
    rng = np.random.default_rng(rows + cols + nt)
    W = rng.integers(0, 256, size=(rows, cols // 2), dtype=np.int32).astype(np.uint8)
    grid = (-(-rows // blk_r), -(-cols // blk_c))
    S = (127 + rng.integers(-6, 3, size=grid)).astype(np.uint8)
    S.flat[0] = 0                                          # 2^-127, a subnormal scale
    S.flat[S.size - 1] = 255                               # NaN
    _KEEP.append((W, S))
    m = dsv4.qmat(W, S, wdt=dsv4.WFP4, cols=cols, blk_r=blk_r, blk_c=blk_c)
    assert gpu.dsv4_gpu_upload(ctypes.byref(m)) == 0
    _check(dsv4, m, _x(rng, nt, cols), ("fp4", rows, cols, nt, blk_r, blk_c))


def test_fp4_scales_off_a_dword(gpu, dsv4):
    """d_s has no alignment rule: scale bytes at any address."""
    import torch
    rows, cols, nt = 40, 1024, 9
    rng = np.random.default_rng(3)
    W = torch.from_numpy(rng.integers(0, 256, size=(rows, cols // 2)).astype(np.uint8)).cuda()
    raw = torch.from_numpy((127 + rng.integers(-6, 3, size=rows * cols // 32 + 4))
                           .astype(np.uint8)).cuda()
    x = torch.from_numpy(rng.standard_normal((nt, cols), dtype=np.float32)).cuda()
    yn = torch.empty(nt, rows, device="cuda")
    y1 = torch.empty(rows, device="cuda")
    for off in range(4):
        s = raw[off:].data_ptr()
        assert gpu.dsv4_gpu_fp4_gemv_n_d(yn.data_ptr(), x.data_ptr(), W.data_ptr(), s, rows, cols,
                                         1, 32, nt, None) == 0
        for t in range(nt):
            assert gpu.dsv4_gpu_fp4_gemv_d(y1.data_ptr(), x[t].data_ptr(), W.data_ptr(), s, rows,
                                           cols, 1, 32, None) == 0
            assert _same(yn[t].cpu().numpy(), y1.cpu().numpy()), (off, t)
