"""Rays at the limits of their fields, through the C ABI.

tmax may be infinite, FLT_MAX or NaN (no limit): such a ray meets what one with a limit far
beyond the scene meets, bit for bit.  The scenes leave nodes with fewer than
four children, whose empty slots are what a limit without a bound could meet.

A component of the direction may be so small that its reciprocal overflows:
the ray meets what the oracle's test of every triangle finds.
"""
import numpy as np
import pytest

import oracle as O
import pppm_amd as P

pytestmark = pytest.mark.gpu

FLT_MAX = np.finfo(np.float32).max


def _scene(kind):
    if kind == "box":
        return P.scenegen(P.SCENE_BOX_CAUSTIC, 1, 6, 8, 8)
    base = P.scenegen(P.SCENE_BOX, 1, 2, 8, 8)
    tri = base.tri[-kind:]  # of one small sphere
    return P.Scene(tri, np.zeros(kind, np.int32), [base.bsdfs[0]], base.lights, base.camera, base.bbox_min,
                   base.bbox_max)


def _rays(tri, n, seed):
    """From inside the box towards triangles, then: every component of the
    direction positive, along an axis, along a plane of two axes."""
    rng = np.random.default_rng(seed)
    c = tri.reshape(-1, 3, 3).mean(axis=1)[np.arange(n) % (len(tri.reshape(-1, 9)))]
    o = rng.uniform(0.1, 4.9, (n, 3))
    d = c - o
    kind = np.arange(n) % 4
    d[kind == 1] = np.abs(d[kind == 1])
    o[kind == 1] = (c - d)[kind == 1]
    for k in range(3):
        cut = ((kind == 2) & (np.arange(n) // 4 % 3 != k)) | ((kind == 3) & (np.arange(n) // 4 % 3 == k))
        d[cut, k] = 0.0
        o[cut, k] = c[cut, k]
    d[np.all(d == 0.0, axis=1), 0] = 1.0
    r = np.zeros(n, P.RAY_DTYPE)
    r["origin"] = o
    r["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r["tmax"] = 1e30
    return r


@pytest.mark.parametrize("builder", [P.BVH_LBVH, P.BVH_PLOC])
@pytest.mark.parametrize("kind", [1, 2, 3, 5, 6, 7, 9, 13, 17, "box"])
def test_a_limit_without_a_bound(gpu_ctx, kind, builder):
    print(f"[case] scene {kind}, builder {builder}", flush=True)
    s = _scene(kind)
    gpu_ctx.upload(s)
    gpu_ctx.build_bvh(builder)
    rays = _rays(np.asarray(s.tri), 6000, 11)
    want = gpu_ctx.intersect(rays)
    hit = want["tri"] >= 0
    assert hit.sum() > 1000
    for tmax in (FLT_MAX, np.float32(np.inf), np.float32(np.nan)):
        r = rays.copy()
        r["tmax"] = tmax
        got = gpu_ctx.intersect(r)
        assert np.array_equal(got["tri"], want["tri"])
        assert np.array_equal(got[hit].view(np.uint32), want[hit].view(np.uint32))
        assert np.array_equal(got["t"][~hit], r["tmax"][~hit], equal_nan=True)
    # the other end: what lies behind the origin counts too
    rays["tmin"] = -1e30
    want = gpu_ctx.intersect(rays)
    for tmin in (-FLT_MAX, np.float32(-np.inf), np.float32(np.nan)):
        r = rays.copy()
        r["tmin"] = tmin
        assert np.array_equal(gpu_ctx.intersect(r).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("tiny", [1e-40, -1e-40, 1.5e-45])
@pytest.mark.parametrize("kind", [3, 5, 17, "box"])
def test_directions_whose_reciprocal_overflows(gpu_ctx, kind, tiny):
    print(f"[case] scene {kind}, components of {tiny}", flush=True)
    s = _scene(kind)
    rays = _rays(np.asarray(s.tri), 6000, 11)
    # about the origin: planes and rays on both sides of zero, whose products
    # with an infinite reciprocal are infinities of both signs
    off = np.float32(2.5)
    tri = (np.asarray(s.tri).reshape(-1, 3) - off).reshape(np.asarray(s.tri).shape)
    s = P.Scene(tri, s.bsdf_id, s.bsdfs, s.lights, s.camera, [v - 2.5 for v in s.bbox_min],
                [v - 2.5 for v in s.bbox_max])
    rays["origin"] -= off
    d = rays["dir"].copy()
    d[d == 0.0] = np.float32(tiny)
    rays["dir"] = d
    gpu_ctx.upload(s)
    gpu_ctx.build_bvh()
    got = gpu_ctx.intersect(rays)["tri"]
    _, ref = O.OracleScene(s).intersect(rays.view(np.float32).reshape(-1, 8), brute=True)
    # a few rays run within a face of a box or along an edge of two triangles
    assert (ref >= 0).sum() > 1000 and (got != ref).sum() <= 0.002 * len(rays)
