"""Where dsv4_gpu_fp8_gemv_n_d keeps the part sums of its split tiles: two
streams never share a place (their calls may overlap on the device), one
stream keeps its own, no memory that a call was given is freed by a later one,
and a captured call has no join, so no address that its graph would keep.
CPU only: an overlap on the device would be a race on that memory."""
import hip_shim

CHILD = r"""
assert L.dsv4_gpu_init() == 0
buf = np.zeros(1 << 12, np.uint8)
a = (buf.ctypes.data + 255) // 256 * 256                     # nothing reads it
names = np.zeros(16, np.uint64)                              # their addresses: the streams

def call(stream, rows, cols, nt, capture=0):
    shim.shim_reset(-1, capture)
    assert L.dsv4_gpu_fp8_gemv_n_d(a, a, a, a, 0, rows, cols, nt, stream) == 0
    return shim.shim_arg1()                                  # the join's part sums

streams = [None] + [names[i:].ctypes.data for i in range(12)]
seen = {}
for rep, (rows, cols, nt) in enumerate([(512, 4096, 16), (1024, 16384, 16), (1536, 7168, 13),
                                        (300, 12288, 9), (2048, 16384, 16), (5376, 12288, 16)]):
    for i, s in enumerate(streams):
        p = call(s, rows, cols, nt)
        assert seen.setdefault(i, p) == p, ("moved", i, rep)
own = sorted(p for p in seen.values() if p)
assert len(set(own)) == len(own), own
# the most: 128 tiles of 2048 x 16384 with four sums each, 336 of 12288 columns with
# three
assert all(b - a >= 4 * max(4 * 16 * 2048, 3 * 16 * 5376) for a, b in zip(own, own[1:])), own
assert shim.shim_frees() == 0
for s in streams[1:]:
    assert call(s, 1536, 7168, 13, capture=1) is None and shim.shim_launches() == 1
print("places", len(own))
"""


def test_part_sums_are_a_streams_own(tmp_path):
    assert hip_shim.run(tmp_path, CHILD).endswith("places 8\n")
