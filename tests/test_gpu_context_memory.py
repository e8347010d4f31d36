"""What a context takes of the device's memory, through the C ABI."""
import ctypes as C

import numpy as np
import pytest

import pppm_amd as P

pytestmark = pytest.mark.gpu

MiB = 1 << 20


def _free():
    hip = C.CDLL("/opt/rocm/lib/libamdhip64.so.7")  # already mapped: the library links it
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.fixture
def ctx():
    with P.Context(0) as c:
        s = P.scenegen(P.SCENE_BOX, 1, 0, 16, 16)
        c.upload(s)
        c.build_bvh()
        c.set_camera(s.camera)
        yield c


@pytest.mark.parametrize("photons", [2000, 131072, 1000000])
def test_record_buffers(ctx, photons):
    print(f"[case] {photons} photons", flush=True)
    before = _free()
    ctx.begin(photons, 1, 0.0866, capacity_factor=2.0)
    used = before - _free()
    # 102 bytes a record of the capacity, 8 a photon; 33 a slot that the photon
    # pass may leave empty: five for each of at most 262,144 paths at a time
    # (256 CUs of 16 waves of 64).  The rest: small buffers, and the allocator,
    # which rounds each up and may reserve some tens of MiB at once for several
    # (up to 19 seen); the slots used to be 139 MB from 131 k photons on
    assert used <= (2 * 102 + 8) * photons + 33 * 5 * min(photons + 255, 262144) + 48 * MiB
    assert ctx.render_pass()["photons_stored"] > 0


def test_counters_of_many_pipelined_passes(ctx):
    # one line of 256 bytes a pass, whatever the copies that its kernels add to
    passes = 4096
    ctx.begin(100, passes + 4, 0.0866)
    ctx.render_passes(4)
    before = _free()
    st = ctx.render_passes(passes)
    assert before - _free() <= 256 * passes + 16 * MiB  # 32 MiB with every copy kept
    assert len(st) == passes and st[-1]["pass_index"] == passes + 4
    # the counts are those of single passes
    ctx.begin(100, 6, 0.0866)
    single = [ctx.render_pass() for _ in range(6)]
    for k in ("photons_stored", "photon_segments", "eye_segments", "hitpoints", "gather_candidates", "gather_inradius"):
        assert [s[k] for s in single[4:]] == [s[k] for s in st[:2]], k


@pytest.mark.parametrize("photons", [20000, 131073, 300001, 700001])
def test_the_slots_hold_a_full_capacity(ctx, photons):
    # waves of 16 to 64 paths on part of the grid and on all of it: with a
    # capacity of just the records, the slots left empty must still fit
    print(f"[case] {photons} photons", flush=True)
    ctx.begin(photons, 1, 0.0866)
    stored = ctx.render_pass()["photons_stored"]
    pos, _, _, key = ctx.last_photons()
    ctx.begin(photons, 1, 0.0866, capacity_factor=(stored - 0.5) / photons)  # the capacity rounds up
    assert ctx.render_pass()["photons_stored"] == stored
    p, _, _, k = ctx.last_photons()
    assert np.array_equal(k, key) and np.array_equal(p, pos)
