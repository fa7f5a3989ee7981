"""Which kernels a batched call takes, at shapes where both were timed, on both
sides of the rules' lines: FP4 and BF16 (us, matrix core / VALU kernel), FP8 with
and without a place for part sums, and the routed experts' host call (batched /
token by token); and whether a single-token FP8 GEMV's x goes through LDS. CPU
only."""
import pytest

import hip_shim

CHILD = r"""
buf = np.zeros(1 << 12, np.uint8)
a = (buf.ctypes.data + 255) // 256 * 256                     # nothing reads it
assert L.dsv4_gpu_init() == 0
def route(call, capture=0):
    shim.shim_reset(-1, capture)
    assert call() == 0
    n = shim.shim_kernel(0)
    assert (b"k_batch_mf" in n) != (b"gemv_n" in n), n
    return b"k_batch_mf" in n
for rows, cols, nt, mf in SHAPES:
    got = route(lambda: CALL(rows, cols, nt))
    assert got == mf, (rows, cols, nt, got)
print("ok")
"""

FP4 = [
    # up to 2048 columns, one VALU workgroup a CU: 6.0 / 4.4, 7.6 / 5.0, 7.9 /
    # 6.5, 8.2 / 8.5, 4.5 / 4.2, 4.5 / 4.8
    (1024, 1024, 4, False), (1024, 1536, 4, False), (64, 1536, 7, False), (2048, 2048, 8, True),
    (2048, 128, 5, False), (2048, 128, 7, True),
    # one tile a CU: 5.8 / 4.7, 5.8 / 6.2, 8.2 / 8.8
    (4096, 512, 4, False), (4096, 512, 7, True), (4096, 2048, 5, True),
    # a round of two a CU begun: 11.1 / 8.3, 10.7 / 7.1, 11.5 / 12.9
    (6144, 1536, 4, False), (6144, 1024, 4, False), (6144, 2048, 6, True),
    # ... and full: 10.6 / 9.1, 10.7 / 11.3, 18.5 / 12.4, 18.6 / 19.3
    (8192, 1024, 5, False), (8192, 1024, 7, True), (16384, 1024, 4, False),
    (16384, 1024, 7, True),
    # above 2048 columns: 15.0 / 12.5, 11.1 / 9.9, 12.5 / 14.6, 15.6 / 18.8
    (1024, 7168, 4, False), (2048, 3584, 4, False), (1024, 4096, 5, True), (2048, 7168, 4, True),
    # scales byte by byte: 12.5 / 11.8, 11.3 / 6.9
    (512, 4128, 5, False), (6144, 1056, 4, False),
]

BF16 = [
    # up to 256 columns; up to 1024: 5.5 / 5.0, 5.7 / 5.4, 5.4 / 5.9; above
    (1024, 256, 2, False), (1024, 256, 3, True),
    (64, 1024, 3, False), (1024, 1024, 3, False), (64, 512, 3, False), (64, 1024, 4, True),
    (256, 4096, 5, False), (256, 4096, 6, True), (256, 7168, 8, False), (256, 7168, 9, True),
    # the widest, ending inside a step or not: 40.3 / 33.1,
    # 43.4 / 42.8, 41.0 / 64.7, 32.1 / 33.0
    (512, 15352, 9, False), (512, 15352, 12, True), (1100, 15352, 9, True),
    (512, 15360, 9, True),
]


@pytest.mark.parametrize("shapes,call", [
    (FP4, "L.dsv4_gpu_fp4_gemv_n_d(a, a, a, a, rows, cols, 1, 32, nt, None)"),
    (BF16, "L.dsv4_gpu_bf16_gemv_n_d(a, a, a, rows, cols, nt, None)")], ids=["fp4", "bf16"])
def test_route(tmp_path, shapes, call):
    child = CHILD.replace("SHAPES", repr(shapes)).replace("CALL(rows, cols, nt)", call)
    assert hip_shim.run(tmp_path, child).endswith("ok\n")


FP8_STREAM = CHILD.split("for rows")[0] + r"""
for rows, cols, nt, eager, captured in SHAPES:
    for sf in (0, 1):
        call = lambda: L.dsv4_gpu_fp8_gemv_n_d(a, a, a, a, sf, rows, cols, nt, a)
        got = route(call), route(call, 1)
        assert got == (eager, captured), (rows, cols, nt, got)
print("ok")
"""

# on a stream with a place for part sums, and captured, where tiles stay whole
# (us, whole tiles / VALU): 14.8 / 13.2, 14.8 / 14.2, 1.16 and 0.77 times, 21.2 /
# 13.4 at 10240 columns, 24.7 / 22.7, 25.2 / 27.9, 27.2 / 24.9, 27.6 / 28.9, 30.8 /
# 29.9, 11.2 / 15.2
FP8_SHAPES = [
    (512, 6144, 5, True, False), (512, 6144, 7, True, True), (512, 4112, 8, True, False),
    (512, 4112, 9, True, True), (64, 11264, 12, True, False), (512, 12288, 12, True, False),
    (512, 12288, 16, True, True), (512, 14336, 8, True, False), (512, 14336, 9, True, True),
    (512, 16384, 9, True, False), (512, 4096, 5, True, True),
    # 64 rows of 192 threads at 10240 columns: E8M0 1.05 times the VALU's at 11
    # tokens, fp32 13.0 / 11.5 at 11, 13.4 / 12.8 at 13
    (64, 10240, 11, False, False), (64, 10240, 13, True, False),
    # tiles that are not split in either: 128 threads a row, 192
    (3000, 7168, 5, True, True), (2000, 12288, 8, True, True), (2000, 12288, 7, False, False),
]


def test_route_fp8(tmp_path):
    child = FP8_STREAM.replace("SHAPES", repr(FP8_SHAPES))
    assert hip_shim.run(tmp_path, child).endswith("ok\n")


MOE = r"""
assert L.dsv4_gpu_init() == 0
def batched(layer, hidden, inter, topk, nt, distinct):
    if not L.dsv4_gpu_has_expert(layer, 0):
        for e in range(64):                                  # nothing reads them
            q = lambda o, r, c: D.DSV4QMat(4096 * (1 + o), 4096 * (4 + o), D.WFP4, r, c, 1, 32)
            ew = D.DSV4ExpertW(q(0, inter, hidden), q(1, inter, hidden), q(2, hidden, inter))
            assert L.dsv4_gpu_bind_expert_d(layer, e, ctypes.byref(ew)) == 0
    idx = np.arange(nt * topk, dtype=np.int32) % distinct
    w = np.ones(nt * topk, np.float32)
    x = np.zeros((nt, hidden), np.float32)
    out = np.empty((nt, hidden), np.float32)
    shim.shim_reset(-1, 0)
    assert L.dsv4_gpu_moe_fp4_n(out.ctypes.data, x.ctypes.data, layer, idx.ctypes.data,
                                w.ctypes.data, nt, topk, hidden, inter, 10.0) == 0
    return any(b"k_mn_prepare" in shim.shim_kernel(i) for i in range(shim.shim_launches()))
for layer, hidden, inter, topk, nt, distinct, want in SHAPES:
    assert batched(layer, hidden, inter, topk, nt, distinct) == want, (hidden, inter, topk, nt)
print("ok")
"""

# layer, hidden, inter, topk, nt, distinct experts, batched: 95.8 / 93.1, 91.3 /
# 88.6, 81.7 / 86.2, 108.0 / 115.9, 51.7 / 61.7, 125.6 / 131.3, shared experts,
# 112.9 / 113.0, 92.1 / 102.2, 91.1 / 93.4
MOE_SHAPES = [
    (0, 7168, 2048, 8, 2, 16, False), (0, 7168, 2048, 7, 2, 14, False),
    (0, 7168, 2048, 6, 2, 12, True), (0, 7168, 2048, 10, 2, 20, True),
    (0, 7168, 2048, 2, 2, 4, True), (0, 7168, 2048, 8, 3, 24, True),
    (0, 7168, 2048, 8, 2, 12, True), (1, 8192, 2048, 8, 2, 16, True),
    (1, 8192, 2048, 6, 2, 12, True), (2, 6144, 2048, 8, 2, 16, True),
]


@pytest.mark.parametrize("mode", [None, "0", "1"])
def test_route_moe(tmp_path, mode):
    shapes = [s if mode is None else s[:-1] + (mode == "0",) for s in MOE_SHAPES]
    env = {} if mode is None else {"DSV4_GPU_MOEN_TOKENWISE": mode}
    assert hip_shim.run(tmp_path, MOE.replace("SHAPES", repr(shapes)), env).endswith("ok\n")


TILES = MOE.split("for layer")[0].replace("range(64)", "range(first, first + n)").replace(
    "def batched(layer,", "def two_tiles(first, n, layer,").replace(
    "layer, 0)", "layer, first)").replace("% distinct", "% distinct + first").replace(
    "k_mn_prepare", "ELi2EEEvPvPKt") + r"""
for layer, (first, n, nt, want) in enumerate(SHAPES):
    assert two_tiles(first, n, layer, 4096, 1024, 8, nt, n) == want, (first, n, nt)
print("ok")
"""

# experts first .. first + n - 1 of a layer, nt tokens of top 8: two column tiles a
# pass where the resident experts average more than five pairs, wherever their ids lie
TILE_SHAPES = [(0, 32, 64, True), (1000, 32, 64, True), (1000, 32, 20, False), (0, 32, 20, False),
               (0, 128, 64, False), (200, 8, 6, True)]


def test_two_tiles_by_experts(tmp_path):
    child = TILES.replace("SHAPES", repr(TILE_SHAPES))
    assert hip_shim.run(tmp_path, child).endswith("ok\n")


GEMV = CHILD.split("def route")[0] + r"""
for rows, cols, sf, xl in SHAPES:
    shim.shim_reset(-1, 0)
    assert L.dsv4_gpu_fp8_gemv_d(a, a, a, a, sf, rows, cols, None) == 0
    n = shim.shim_kernel(0)
    assert n.split(b"k_fp8_gemvILi")[1].split(b"E")[4] == b"Li%d" % xl, (rows, cols, sf, n)
print("ok")
"""

# rows, cols, scales, the waves of a row whose x goes through LDS or 0 (us, cold, own
# loads / through LDS): 4.01 / 4.20, 4.69 / 4.86, 7.02 / 6.64, 14.5 / 12.2, 7.4 / 6.8,
# 8.40 / 8.60, 5.99 / 5.57, 11.7 / 12.0, 6.63 / 6.30, 10.05 / 9.67, 9.60 / 10.10
GEMV_SHAPES = [
    (78, 15680, 1, 0), (199, 15664, 0, 0), (936, 14400, 0, 4), (4096, 13312, 1, 4),
    (1024, 16384, 0, 4), (5823, 5200, 1, 0), (20000, 5200, 1, 2), (4096, 4096, 0, 1),
    (7168, 7168, 0, 0), (2048, 8192, 0, 2), (4435, 7104, 0, 2), (5786, 6240, 0, 0),
]


def test_x_through_lds(tmp_path):
    child = GEMV.replace("SHAPES", repr(GEMV_SHAPES))
    assert hip_shim.run(tmp_path, child).endswith("ok\n")
