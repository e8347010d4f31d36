"""The quad traversal at the sizes where its waves, slots and leaves end,
through the C ABI.

A ray's hit does not depend on the rays traced beside it, so the first n rays
of a batch alone hit what they hit in the whole batch, bit for bit; the whole
batch, rays with an interval of their own, leaves of one and two triangles and
eye passes of odd sizes are held against the oracle.
"""
import numpy as np
import pytest

import oracle as O
import pppm_amd as P

pytestmark = pytest.mark.gpu


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    r = np.zeros(n, P.RAY_DTYPE)
    r["origin"] = rng.uniform(0.1, 4.9, (n, 3))
    d = rng.normal(size=(n, 3))
    r["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r["tmax"] = 1e30
    return r


@pytest.fixture(scope="module")
def box(gpu_ctx):
    s = P.scenegen(P.SCENE_BOX_CAUSTIC, 1, 12, 16, 16)
    gpu_ctx.upload(s)
    gpu_ctx.build_bvh()
    rays = _rays(300001, 5)
    return gpu_ctx, s, rays, gpu_ctx.intersect(rays)


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 31, 63, 64, 65, 255, 257, 4097, 65535, 65537, 262145])
def test_a_part_of_a_batch_hits_the_same(box, n):
    ctx, _, rays, hits = box
    print(f"[case] {n} rays", flush=True)
    assert np.array_equal(ctx.intersect(rays[:n]).view(np.uint32), hits[:n].view(np.uint32))


def test_rays_with_an_interval_match_the_oracle(box):
    ctx, s, rays, hits = box
    n = 6000
    r = rays[:n].copy()
    # from just behind the first hit, to a limit that cuts some of the second ones off
    r["tmin"] = hits["t"][:n] * np.float32(1.001) + np.float32(1e-3)
    r["tmax"] = np.random.default_rng(2).uniform(1.0, 8.0, n)
    got = ctx.intersect(r)
    t, tri = O.OracleScene(s).intersect(r.view(np.float32).reshape(-1, 8), brute=True)
    # hit or miss may differ only where a distance rounds to the other side of the interval
    same = (got["tri"] >= 0) == (tri >= 0)
    assert same.mean() > 0.999
    both = (got["tri"] >= 0) & (tri >= 0)
    close = np.abs(got["t"][both] - t[both]) <= 2e-5 * t[both] + 2e-6
    assert both.sum() > 100 and close.mean() > 0.999
    assert np.all(got["t"][got["tri"] < 0] == r["tmax"][got["tri"] < 0])


@pytest.mark.parametrize("builder", [P.BVH_LBVH, P.BVH_PLOC])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 17])
def test_leaves_of_few_triangles(gpu_ctx, n, builder):
    print(f"[case] {n} triangles, builder {builder}", flush=True)
    base = P.scenegen(P.SCENE_BOX, 1, 2, 8, 8)
    tri = base.tri[-n:]  # triangles of one small sphere: leaves fill up
    sub = P.Scene(tri, np.zeros(n, np.int32), [base.bsdfs[0]], base.lights, base.camera, base.bbox_min, base.bbox_max)
    gpu_ctx.upload(sub)
    gpu_ctx.build_bvh(builder)
    rays = _rays(5000, n)
    c = tri.reshape(-1, 3, 3).mean(axis=1)[np.arange(5000) % n]  # towards a triangle each
    d = c - rays["origin"]
    rays["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    got = gpu_ctx.intersect(rays)
    t, ref = O.OracleScene(sub).intersect(rays.view(np.float32).reshape(-1, 8), brute=True)
    assert np.array_equal(got["tri"] >= 0, ref >= 0)
    hit = ref >= 0
    assert (got["tri"][hit] == ref[hit]).mean() > 0.999
    # t is interpolated with the edge functions, whose rounding (2^-24 of the
    # distance) against the triangle's projected size moves it by about
    # 2^-21 t tan(angle to the normal): these rays graze small triangles
    v = tri.reshape(-1, 3, 3).astype(np.float64)[ref[hit]]
    nrm = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    cos = np.abs(np.sum(nrm * rays["dir"][hit], axis=1)) / np.linalg.norm(nrm, axis=1)
    assert np.all(np.abs(got["t"][hit] - t[hit]) <= 2e-5 * t[hit] / cos + 2e-6)


@pytest.mark.parametrize("w,h", [(1, 1), (3, 5), (16, 1), (17, 1), (64, 1), (65, 3), (131, 67), (520, 300)])
def test_eye_pass_of_odd_sizes(gpu_ctx, w, h):
    print(f"[case] eye pass {w} x {h}", flush=True)
    s = P.scenegen(P.SCENE_BOX_CAUSTIC, 1, 6, w, h)
    gpu_ctx.upload(s)
    gpu_ctx.build_bvh()
    gpu_ctx.set_camera(s.camera)
    gpu_ctx.begin(1000, 1, 0.0866, ray_eps=1e-4)
    gpu_ctx.render_pass()
    pos, _, wt, pix = gpu_ctx.last_hitpoints()
    has, op, _, ow, _ = O.OracleScene(s).eye_pass(s.camera, 1, 1e-4, 0x7A75)
    g = np.zeros_like(has)
    g[pix] = 1
    assert len(np.unique(pix)) == len(pix)
    # paths through glass decide reflection in 32 and 64 bits
    assert (g != has).sum() <= max(1, 0.002 * w * h)
    sel = has[pix] == 1
    near = np.abs(pos[sel] - op[pix[sel]]).max(axis=1) < 1e-3
    assert (~near).sum() <= max(1, 0.002 * w * h)
    # the weight divides by the Fresnel factor picked, whose slope has no bound
    # at grazing angles: position rounding may show in a few pixels seen through
    # the curved glass
    a, b = wt[sel][near].astype(np.float64), ow[pix[sel]][near]
    close = np.all(np.abs(a - b) <= 1e-4 * np.abs(b) + 1e-6, axis=1)
    assert (~close).sum() <= max(1, 0.001 * w * h)
