"""The Hachisuka update of a few render points, through the C ABI, against a
loop over the photons in double: eight lanes take a point, so images of fewer
than eight points and of a few more end inside and at the ends of a wave.

The loop takes the device's own photons and hit points (those of a plain pass
with the same seed are the same) in the fixed order of the update: a point's
buckets in z, y, x order of its cells, each in photon order, every photon held
against the radius that the ones before it left.  With the same FP32 inputs
each decision is the same, and the results agree to double rounding.  The
camera's narrow field keeps the radius, which follows the hit points' extent,
small against the scene.
"""
import numpy as np
import pytest

import oracle as O
import pppm_amd as P

pytestmark = pytest.mark.gpu

PHOTONS, PASSES, ALPHA, R1, SEED = 60000, 2, 0.7, 0.0866, 0x7A75


def _cell(x, mn, scale):
    return np.abs(((x - mn) * scale).astype(np.int32))


def _hash(c, size):
    c = c.astype(np.uint32)
    with np.errstate(over="ignore"):
        return int((c[0] * np.uint32(73856093) ^ c[1] * np.uint32(19349663) ^ c[2] * np.uint32(83492791)) %
                   np.uint32(size))


def _update(state, x, nx, w, irad, bmin, pos, flux, nrm, cs, ce, sidx):
    r2, n, f = state
    if n == 0:
        r2, f = irad * irad, np.zeros(3)
    mn, scale = bmin - irad, 1.0 / (2.0 * irad)
    lo = _cell(x - irad, mn, scale)
    hi = np.minimum(_cell(x + irad, mn, scale), lo + 1)
    seen = []
    for iz in range(lo[2], hi[2] + 1):
        for iy in range(lo[1], hi[1] + 1):
            for ix in range(lo[0], hi[0] + 1):
                h = _hash(np.array([ix, iy, iz]), len(cs))
                if h in seen:
                    continue
                seen.append(h)
                for j in sidx[cs[h]:ce[h]]:
                    d = x - pos[j]
                    if not (nrm[j] @ nx > 0.0 and d @ d <= r2):
                        continue
                    na = n * ALPHA
                    g = (na + ALPHA) / (na + 1.0)
                    r2 *= g
                    n += 1
                    f = (f + w * flux[j]) * g
    return r2, n, f


@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (3, 1), (1, 7), (8, 1), (3, 3), (5, 7)])
def test_few_points_match_a_loop_over_the_photons(gpu_ctx, w, h):
    print(f"[case] {w} x {h}", flush=True)
    s = P.scenegen(P.SCENE_BOX, 1, 2, w, h)
    s.camera.fov_y_deg = 4.0
    bmin = np.asarray(s.tri, np.float32).reshape(-1, 3).min(axis=0).astype(np.float64)
    gpu_ctx.upload(s)
    gpu_ctx.build_bvh()
    gpu_ctx.set_camera(s.camera)
    gpu_ctx.begin(PHOTONS, PASSES, R1, alpha=ALPHA, seed=SEED)
    passes = []
    for _ in range(PASSES):
        gpu_ctx.render_pass()
        passes.append((gpu_ctx.last_photons(), gpu_ctx.last_hitpoints()))
    gpu_ctx.begin(PHOTONS, PASSES, R1, alpha=ALPHA, seed=SEED, method=P.METHOD_HACHISUKA)
    state = [(0.0, 0, np.zeros(3)) for _ in range(w * h)]
    for (pos, flux, nrm, _), (hp, hn, hw, pix) in passes:
        st = gpu_ctx.render_pass()
        assert st["hitpoints"] == len(pix) > 0 and st["photons_stored"] == len(pos)
        ext = (hp.max(axis=0).astype(np.float64) - hp.min(axis=0)).sum() / 3.0
        irad = st["radius"]
        assert irad == (R1 if len(pix) == 1 else pytest.approx(ext / ((w + h) / 2.0) * 8.0, rel=1e-12))
        # a bucket holds its photons in their order, as the records come
        sidx, cs, ce = O.hashgrid_points(pos, st["hash_size"], 1.0 / (2.0 * irad), bmin - irad)
        for j in (0, len(pos) // 2, len(pos) - 1):
            b = _hash(_cell(pos[j].astype(np.float64), bmin - irad, 1.0 / (2.0 * irad)), len(cs))
            assert j in sidx[cs[b]:ce[b]]
        p64, f64, n64 = pos.astype(np.float64), flux.astype(np.float64), nrm.astype(np.float64)
        before = sum(c[1] for c in state)
        for k, i in enumerate(pix):
            state[i] = _update(state[i], hp[k].astype(np.float64), hn[k].astype(np.float64), hw[k].astype(np.float64),
                               irad, bmin, p64, f64, n64, cs, ce, sidx)
        assert st["gather_inradius"] == sum(c[1] for c in state) - before > 0
    want = np.array([f / (np.pi * r2) if n else f for r2, n, f in state]) / PASSES
    np.testing.assert_allclose(gpu_ctx.image().reshape(-1, 3), want, rtol=1e-10, atol=1e-300)
