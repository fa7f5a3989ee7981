"""A kernel launch that fails is reported: every batched GEMV entry point on
device buffers returns -1 for it, whichever of its launches it is. CPU only."""
import pytest

import hip_shim

CHILD = r"""
buf = np.zeros(1 << 12, np.uint8)
a = (buf.ctypes.data + 255) // 256 * 256                     # nothing reads it
# 8200 x 512 from 5 tokens on: the f32 matrix core; below: the VALU kernels.
# 512 x 4096 at 16 tokens: tiles split over workgroups, with a join
calls = []
for nt in (1, 2, 5, 17, 64):
    for sf in (0, 1):
        calls.append(lambda nt=nt, sf=sf: L.dsv4_gpu_fp8_gemv_n_d(
            a, a, a, a, sf, 8200, 512, nt, None))
    calls.append(lambda nt=nt: L.dsv4_gpu_bf16_gemv_n_d(a, a, a, 8200, 512, nt, None))
    calls.append(lambda nt=nt: L.dsv4_gpu_fp4_gemv_n_d(a, a, a, a, 8200, 512, 1, 32, nt, None))
calls.append(lambda: L.dsv4_gpu_fp8_gemv_n_d(a, a, a, a, 0, 512, 4096, 16, None))
assert L.dsv4_gpu_init() == 0
most = 0
for i, call in enumerate(calls):
    shim.shim_reset(-1, 0)
    assert call() == 0 and shim.shim_launches() >= 1, i
    n = shim.shim_launches()
    most = max(most, n)
    for at in range(n):
        shim.shim_reset(at, 0)
        assert call() == -1, (i, at)
print("most launches", most)
"""


@pytest.mark.parametrize("env,most", [({}, 2), ({"DSV4_GPU_MFN_L": "16"}, 1),
                                      ({"DSV4_GPU_FP8_MFN": "0"}, 1)])
def test_failed_launch_is_reported(tmp_path, env, most):
    assert hip_shim.run(tmp_path, CHILD, env).endswith("most launches %d\n" % most)
