"""Results written to pinned memory of the caller, through the C ABI: the same
bits as in pageable memory, at sizes about the ends of the 1 MiB buffers that
pageable memory takes."""
import ctypes as C

import numpy as np
import pytest

import pppm_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 65535, 65536, 65537, 200000])
def test_hits_in_pinned_memory(gpu_ctx, n):
    print(f"[case] {n} rays", flush=True)
    s = P.scenegen(P.SCENE_BOX, 1, 4, 8, 8)
    gpu_ctx.upload(s)
    gpu_ctx.build_bvh()
    rng = np.random.default_rng(n)
    rays = np.zeros(n, P.RAY_DTYPE)
    rays["origin"] = rng.uniform(0.5, 4.5, (n, 3))
    rays["dir"] = rng.normal(size=(n, 3))
    rays["tmax"] = 1e30
    want = gpu_ctx.intersect(rays)
    hip = C.CDLL("/opt/rocm/lib/libamdhip64.so.7")  # already mapped: the library links it
    mem = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(mem), C.c_size_t(16 * n + 16), C.c_uint(0)) == 0
    try:
        out = np.ctypeslib.as_array(C.cast(mem, C.POINTER(C.c_uint8)), (16 * n + 16,))
        out[:] = 7
        assert P.lib().pppm_intersect(gpu_ctx.h, rays.ctypes.data, n, mem) == P.OK
        assert np.array_equal(out[:16 * n], want.view(np.uint8).reshape(-1))
        assert np.all(out[16 * n:] == 7)
    finally:
        hip.hipHostFree(mem)
