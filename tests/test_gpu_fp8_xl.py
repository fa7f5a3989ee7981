"""The single-token FP8 GEMV with x through LDS (csrc/dsv4_fp8.hip) at the
edges of its rounds of 1024 columns: rows of 1 to 64 threads and of 65 to 256,
x that ends inside a round, and rows that end inside a workgroup's step. x
straight from memory and through LDS are the same arithmetic, so their bits
are equal; against 64 bits the error is that of a sum of `cols` products in
f32, bounded by cols * 2^-24 of the sum of their magnitudes."""
import ctypes

import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu

_KEEP = []          # resident matrices are keyed by host address


@pytest.mark.parametrize("scales", ["e8m0", "f32"])
@pytest.mark.parametrize("rows,cols", [
    (1, 16), (5, 48), (700, 512), (130, 1008), (64, 1024), (67, 1040), (1025, 1536),
    (259, 2032), (2100, 2048), (33, 2064), (70, 4096), (66, 4112), (1300, 7168), (37, 8192),
    (41, 12304), (35, 16368), (300, 16384)])
def test_x_through_lds(gpu, dsv4, monkeypatch, rows, cols, scales):
    rng = np.random.default_rng(rows * 31 + cols)
    W = common.fp8_codes(rng, (rows, cols))
    Sf, Se = common.fp8_scales(rng, rows, cols)
    S = Se if scales == "e8m0" else Sf
    _KEEP.append((W, S))
    m = dsv4.qmat(W, S)
    up = gpu.dsv4_gpu_upload if scales == "e8m0" else gpu.dsv4_gpu_upload_f32s
    assert up(ctypes.byref(m)) == 0
    x = rng.standard_normal(cols, dtype=np.float32)
    got = {}
    for xl in ("0", "1"):
        for r in ("1", "4"):
            monkeypatch.setenv("DSV4_GPU_FP8_XL", xl)
            monkeypatch.setenv("DSV4_GPU_FP8_R", r)
            got[xl, r] = dsv4.mmq(m, x).copy()
    for y in got.values():
        assert common.bits_equal(y, got["0", "1"])
    s = np.repeat(np.repeat(Sf.astype(np.float64), 128, 0)[:rows], 128, 1)[:, :cols]
    p = common.e4m3_table()[W].astype(np.float64) * s * x
    assert np.all(np.abs(got["1", "1"] - p.sum(1)) <= cols * 2.0 ** -24 * np.abs(p).sum(1))


# rows of 64, 128, 192 and 256 threads, x filling its last round of 1024 columns
# or not, one step per workgroup and several
@pytest.mark.parametrize("scales", ["e8m0", "f32"])
@pytest.mark.parametrize("rows,cols", [
    (300, 1536), (256, 4608), (1536, 4608), (2100, 6144), (5130, 7168), (200, 8192),
    (259, 9216), (1100, 12288), (256, 13312), (600, 13312), (260, 16384), (5000, 16384)])
def test_rule_and_prefetch(gpu, dsv4, monkeypatch, rows, cols, scales):
    """The launch rule's own choice and every form it chooses from (x's way,
    rows per step, prefetch) give the same bits."""
    rng = np.random.default_rng(rows * 37 + cols)
    W = common.fp8_codes(rng, (rows, cols))
    Sf, Se = common.fp8_scales(rng, rows, cols)
    S = Se if scales == "e8m0" else Sf
    _KEEP.append((W, S))
    m = dsv4.qmat(W, S)
    up = gpu.dsv4_gpu_upload if scales == "e8m0" else gpu.dsv4_gpu_upload_f32s
    assert up(ctypes.byref(m)) == 0
    x = rng.standard_normal(cols, dtype=np.float32)
    want = dsv4.mmq(m, x).copy()
    for xl in ("0", "1"):
        for r in ("1", "2", "4"):
            for pf in ("0", "1"):
                monkeypatch.setenv("DSV4_GPU_FP8_XL", xl)
                monkeypatch.setenv("DSV4_GPU_FP8_R", r)
                monkeypatch.setenv("DSV4_GPU_FP8_PF", pf)
                assert common.bits_equal(dsv4.mmq(m, x), want), (xl, r, pf)
