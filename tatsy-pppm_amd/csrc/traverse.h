// traverse.h -- closest-hit traversal of the 4-wide BVH (device code).
//
// Four lanes (a quad) trace one ray, sixteen rays per wave at a time.  In a
// node step lane c of the quad tests child c: two 16-byte loads of its 32
// bytes of the node's 128-byte line, one slab test, and its place among the
// children by comparing keys across the quad (DPP); in a leaf step lanes 0 and
// 1 test a triangle each.  The wave's 64 lanes own one ray each: the rays wait in
// LDS, a quad whose ray is finished takes the next waiting one, and the owner
// reads the hit from its slot.  What bounds it is VALU issue and, for the last
// rays of a wave, the latency of the chain of node fetches: with one ray per
// lane the four slab tests and the sort ran in every lane with 13 of 64 lanes
// busy on average; here a step is half as long and the lanes it occupies do
// work.  Photon pass of the caustic box (0.7 M triangles, 8.9 M rays), a pass by
// itself: 4.2 ms with one ray per lane, 3.1 ms with a quad per ray; 0.91 -> 0.77 ms
// on 60 k triangles, 0.38 -> 0.26 ms at 200 k photons, 0.30 -> 0.16 ms at 10 k.  What
// is left is the latency of node fetches: a step waits for the slowest of up to
// sixteen, and four in ten miss the 4 MiB L2 of their die.
// The loop is the while-while form with postponed leaves of Aila and Laine
// (2009): a quad that reaches its first leaf keeps it waiting and goes on
// through inner nodes until most quads of the wave have one.
#pragma once

#include "pppm_device.h"

// Entries a traversal can leave on its stack at most: three per level below
// the root and the root's own place; a stack has as many in LDS as its tree
// needs (SceneDev::stack), so there is nothing to spill.
#define STACK_MAX 128

// Conservative slab test (Ize 2013): the exit distance is scaled up by
// 1 + 2^-22 so FP32 rounding cannot cull a box the triangle test would hit.
#define SLAB_FAR_SCALE 1.00000024f

// Per-lane traversal work, counted by the COUNT instantiation only.
struct TravCount {
    uint32_t nodes = 0;  // inner nodes visited (one 128-byte fetch each)
    uint32_t tris = 0;   // triangles tested (48 bytes each)
};

typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// Word 3 of a raw buffer resource on CDNA: 32-bit data format, no swizzle.
#define BUFFER_RSRC_WORD3 0x00020000

#define QUADS 16  // rays a wave traces at a time
// what a quad leaves in the last word of a finished ray's slot (never an axis code)
#define RAY_DONE 0xFFFFFFFFu

// LDS of one wave: 64 ray slots of three 16-byte words, laid out [word][slot];
// the ring of waiting slots; the quads' stacks, laid out [entry][quad].
//   waiting: (o, shear x) (1 / d, shear y) (tmin, tmax, shear z, axis code)
//   traced:  (t, triangle, u, v) -          (-, -, -, RAY_DONE once finished)
struct WaveRays {
    float4* slot;
    uint8_t* ring;
    char* stack;  // this lane's quad: entry k STACK_STEP * k bytes in
};
#define STACK_STEP (4 * QUADS)
__host__ __device__ inline uint32_t wave_rays_bytes(int32_t stack) {
    return 3 * 64 * 16 + 64 + (uint32_t)stack * STACK_STEP;
}
__device__ inline WaveRays wave_rays(char* block_lds, int32_t stack) {
    char* p = block_lds + (threadIdx.x >> 6) * wave_rays_bytes(stack);
    WaveRays w;
    w.slot = reinterpret_cast<float4*>(p);
    w.ring = reinterpret_cast<uint8_t*>(p + 3 * 64 * 16);
    w.stack = p + 3 * 64 * 16 + 64 + (threadIdx.x & 60);
    return w;
}

// A quad's ray (the same values in its four lanes): the watertight test's
// shear, the slab test's scaled inverse direction, and how far it has got.
struct QuadRay {
    RayPre pre;  // pre.o is the origin
    float ix, iy, iz, ox, oy, oz;
    float tmin, t;  // t: the closest hit so far
    float t_far;    // slab_limit(t)
    int32_t cur;    // the next inner node (>= 0), a leaf root (< 0), or EMPTY_REF: no ray
    int32_t sp;     // bytes of the stack in use; the lowest entry is EMPTY_REF
    int32_t slot;   // whose ray it is
};

// What a box's entry distance is held against for a closest hit at t: never
// infinite, so that an empty slot, entered at infinity, is missed also by a ray
// without a limit (t infinite, so near the largest float that scaling it
// overflows, or NaN).
__device__ inline float slab_limit(float t) { return fminf(t * SLAB_FAR_SCALE, 3.402823466e+38f); }

// The wave's waiting rays: ring positions [head, tail), the same in every lane.
struct RayQueue {
    uint32_t head = 0, tail = 0;
};

// Puts the rays of the lanes with `put` set in line.  Called by the whole wave.
__device__ inline void rays_put(const WaveRays& w, RayQueue& rq, bool put, v3f o, v3f d, float tmin, float tmax) {
    const int lane = threadIdx.x & 63;
    const uint64_t m = __ballot(put);
    if (put) {
        // inverse direction as the reference computes it (qbvh_accel.cc:219-221)
        const float ix = d.x == 0.0f ? 1.0e20f : 1.0f / d.x;
        const float iy = d.y == 0.0f ? 1.0e20f : 1.0f / d.y;
        const float iz = d.z == 0.0f ? 1.0e20f : 1.0f / d.z;
        const RayPre p = ray_pre(o, d, mk(ix, iy, iz));
        w.slot[lane] = make_float4(o.x, o.y, o.z, p.sx);
        w.slot[64 + lane] = make_float4(ix, iy, iz, p.sy);
        w.slot[128 + lane] =
            make_float4(tmin, tmax, p.sz, __uint_as_float((uint32_t)(p.kx | (p.ky << 2) | (p.kz << 4))));
        w.ring[(rq.tail + (uint32_t)__popcll(m & lanemask_lt())) & 63u] = (uint8_t)lane;
    }
    rq.tail += (uint32_t)__popcll(m);
    wave_lds_fence();
}

// Whether the ray this lane put has been traced.
__device__ inline bool ray_done(const WaveRays& w) {
    return __float_as_uint(w.slot[128 + (threadIdx.x & 63)].w) == RAY_DONE;
}
// Its hit.
__device__ inline Hit ray_hit(const WaveRays& w) {
    const float4 h = w.slot[threadIdx.x & 63];
    Hit r;
    r.t = h.x;
    r.tri = __float_as_int(h.y);
    r.u = h.z;
    r.v = h.w;
    return r;
}

// Traces until at most `keep` of the wave's rays are unfinished (waiting or in
// a quad; keep = 0: none).  Called by the whole wave; q.cur = EMPTY_REF before
// the first call.
// ZERO_TMIN: every ray was put with tmin = 0.
template <bool COUNT, bool ZERO_TMIN>
__device__ inline void rays_trace(const SceneDev& sc, const WaveRays& w, QuadRay& q, RayQueue& rq, int keep,
                                  TravCount* tc) {
    const int lane = threadIdx.x & 63;
    const int c = lane & 3;
    const uint64_t quads_before = ~(~0ull << (lane & ~3));  // lanes of the quads before this one
    const uint32_t nearer_slot = 3u - (uint32_t)c, miss_key = 0x80000000u | (uint32_t)c;
#define STACK(at) (*reinterpret_cast<int32_t*>(w.stack + (at)))
#define POP() (q.sp -= STACK_STEP, STACK(q.sp))
    // the node array as a buffer: 32-bit per-lane byte offsets, and a fetch
    // past its end reads zeros instead of faulting
    const __amdgpu_buffer_rsrc_t nbuf = __builtin_amdgcn_make_buffer_rsrc(
        (void*)sc.nodes, (short)0, sc.n_nodes * (int32_t)sizeof(Node4), BUFFER_RSRC_WORD3);
    while (true) {
        // quads without a ray take the next waiting ones
        if (rq.head != rq.tail) {
            const uint64_t idle = __ballot(q.cur == (int32_t)EMPTY_REF);
            const uint32_t r = (uint32_t)__popcll(idle & quads_before) >> 2;
            const uint32_t waiting = rq.tail - rq.head;
            if (q.cur == (int32_t)EMPTY_REF && r < waiting) {
                const int s = w.ring[(rq.head + r) & 63u];
                const float4 a = w.slot[s], b = w.slot[64 + s], e = w.slot[128 + s];
                const uint32_t code = __float_as_uint(e.w);
                q.slot = s;
                q.pre.o = xyz(a);
                q.pre.sx = a.w;
                q.pre.sy = b.w;
                q.pre.sz = e.z;
                q.pre.kx = (int)(code & 3u);
                q.pre.ky = (int)((code >> 2) & 3u);
                q.pre.kz = (int)(code >> 4);
                q.ix = b.x;
                q.iy = b.y;
                q.iz = b.z;
                q.ox = a.x * b.x;
                q.oy = a.y * b.y;
                q.oz = a.z * b.z;
                q.tmin = e.x;
                q.t = e.y;
                q.t_far = slab_limit(e.y);
                q.cur = sc.root;
                q.sp = STACK_STEP;
                wave_lds_fence();
                if (c == 0) {
                    STACK(0) = EMPTY_REF;
                    // until a triangle is hit: a miss
                    w.slot[s] = make_float4(e.y, __int_as_float(-1), 0.0f, 0.0f);
                    if (sc.root == (int32_t)EMPTY_REF) w.slot[128 + s].w = __uint_as_float(RAY_DONE);
                }
                wave_lds_fence();
            }
            rq.head += min(waiting, (uint32_t)__popcll(idle) >> 2);
        }
        const uint64_t busy = __ballot(q.cur != (int32_t)EMPTY_REF);
        const int unfinished = (int)(__popcll(busy) >> 2) + (int)(rq.tail - rq.head);
        if (unfinished <= keep) break;
        const bool mine = q.cur != (int32_t)EMPTY_REF;
        // cur: an inner node or EMPTY_REF (the stack is empty); leaf: a leaf
        // waiting for its triangle tests (< 0) or none
        int32_t leaf = EMPTY_REF;
        if (q.cur < 0) {  // a leaf root
            leaf = q.cur;
            q.cur = POP();
        }
        // inner nodes, until the quads with a leaf waiting are more than twice
        // those that still look for one (a photon pass takes 16 % longer waiting
        // for the last quad, 3 and 6 % at once and five times; with few rays the
        // ratio does not matter)
        while (true) {
            const bool inner = (uint32_t)q.cur < (uint32_t)EMPTY_REF;
            const int stepping = (int)__popcll(__ballot(inner && leaf >= 0));
            if (stepping == 0 || 2 * stepping < (int)__popcll(__ballot(leaf < 0))) break;
            if (inner) {
                if (COUNT && c == 0) tc->nodes++;
                const int at = (int)(((uint32_t)q.cur << 7) | ((uint32_t)c << 5));
                const v4u p = __builtin_amdgcn_raw_buffer_load_b128(nbuf, at, 0, 0);
                const v4u r = __builtin_amdgcn_raw_buffer_load_b128(nbuf, at, 16, 0);
                // the near and the far plane of each axis by the direction's sign: an
                // axis whose products are infinities of both signs (a direction
                // component whose reciprocal overflows) has a NaN for a plane,
                // which must not limit the interval, while min and max of the two
                // planes would take the other one for both
                const bool fx = q.ix >= 0.0f, fy = q.iy >= 0.0f, fz = q.iz >= 0.0f;
                const float x0 = __uint_as_float(fx ? p.x : p.w) * q.ix - q.ox;
                const float x1 = __uint_as_float(fx ? p.w : p.x) * q.ix - q.ox;
                const float y0 = __uint_as_float(fy ? p.y : r.x) * q.iy - q.oy;
                const float y1 = __uint_as_float(fy ? r.x : p.y) * q.iy - q.oy;
                const float z0 = __uint_as_float(fz ? p.z : r.y) * q.iz - q.oz;
                const float z1 = __uint_as_float(fz ? r.y : p.z) * q.iz - q.oz;
                const float n = fmaxf(fmaxf(x0, y0), fmaxf(z0, ZERO_TMIN ? 0.0f : q.tmin));
                const float f = fminf(fminf(x1, y1), z1);
                // rays that bring their own limits: without one at the near end (tmin
                // -inf or NaN) an empty slot may be entered at -inf, and f is NaN where
                // every component's reciprocal overflows.  Two comparisons where
                // neither can be: one against the smaller of the two limits made the
                // path that ends a pass of an open scene 2 % longer
                const bool hit = ZERO_TMIN ? n <= f * SLAB_FAR_SCALE && n <= q.t_far
                                           : n <= fminf(f * SLAB_FAR_SCALE, q.t_far) && n > -__builtin_inff();
                // the children hit go on the stack farthest first, the nearest
                // on top, which is taken next; the missed ones above it, where
                // they do not count.  So lane c writes its child at the number
                // of keys below its own: the complement of the entry distance
                // (non-negative, so its bits order like the value) with the
                // child slot in the two low bits, above all of them for a miss
                const uint32_t key =
                    hit ? ((~__float_as_uint(n) & 0x7FFFFFFCu) | nearer_slot) : miss_key;
                const uint32_t k1 = (uint32_t)quad_read<QUAD_NEXT1>((int32_t)key);
                const uint32_t k2 = (uint32_t)quad_read<QUAD_NEXT2>((int32_t)key);
                const uint32_t k3 = (uint32_t)quad_read<QUAD_NEXT3>((int32_t)key);
                const int place = (k1 < key ? 1 : 0) + (k2 < key ? 1 : 0) + (k3 < key ? 1 : 0);
                STACK(q.sp + place * STACK_STEP) = (int32_t)r.z;
                int pushed = hit ? STACK_STEP : 0;
                pushed += quad_read<QUAD_XOR1>(pushed);
                pushed += quad_read<QUAD_NEXT2>(pushed);
                q.sp += pushed;
                wave_lds_fence();
                // the first leaf waits and traversal goes on with the entry
                // below it (both read at once; below the lowest entry lies
                // something else, which is read but not taken)
                const int32_t top = STACK(q.sp - STACK_STEP), below = STACK(q.sp - 2 * STACK_STEP);
                wave_lds_fence();
                const bool waits = top < 0 && leaf >= 0;
                q.cur = waits ? below : top;
                leaf = waits ? top : leaf;
                q.sp -= waits ? 2 * STACK_STEP : STACK_STEP;
            }
        }
        // the waiting leaf, then a leaf popped behind it: lane c its triangle
        // c, with the outcome of testing one after the other
        while (leaf < 0) {
            const uint32_t v = (uint32_t)(~leaf);
            const int32_t tri = (int32_t)(v >> 3) + c;
            const int32_t cnt = (int32_t)(v & 7u) + 1;
            if (COUNT && c == 0) tc->tris += (uint32_t)cnt;
            TriHit h;
            h.t = 0.0f;
            bool met = false;
            if (c < cnt) {
                const float4* tp = sc.tris + 3 * (int64_t)tri;
                met = tri_watertight(q.pre, tp[0], tp[1], tp[2], q.tmin, h);
            }
            // lane 1 is held against what lane 0 leaves
            const float t0 = __int_as_float(
                quad_read<QUAD_LANE0>(__float_as_int(met && tri_nearer(h, q.t) ? h.t : q.t)));
            const bool wins = met && tri_nearer(h, c == 0 ? q.t : t0);
            const uint32_t won = (uint32_t)(__ballot(wins) >> (lane & ~3)) & 3u;
            if (won != 0u) {
                q.t = won & 2u ? __int_as_float(quad_read<QUAD_LANE1>(__float_as_int(h.t))) : t0;
                q.t_far = slab_limit(q.t);
                if (c == (int)(won >> 1)) w.slot[q.slot] = make_float4(h.t, __int_as_float(tri), h.u, h.v);
            }
            leaf = q.cur;
            if (q.cur < 0) q.cur = POP();
        }
        if (mine && q.cur == (int32_t)EMPTY_REF && c == 0) w.slot[128 + q.slot].w = __uint_as_float(RAY_DONE);
        wave_lds_fence();
    }
#undef POP
#undef STACK
}

// Rays a wave owns at a time where `rays` rays are shared out to `waves` waves
// that are all resident: a multiple of the sixteen it traces at a time, so that
// few rays spread over the chip, one per quad, and many fill the 64 slots.
inline int wave_ray_slots(int64_t rays, int64_t waves) {
    const int64_t per = (rays + waves - 1) / waves;
    return (int)(per <= QUADS ? QUADS : per >= 64 ? 64 : (per + QUADS - 1) / QUADS * QUADS);
}

// A leaf-order triangle's record.
struct TriRec {
    float4 a, b, c;
};
__device__ inline TriRec tri_record(const SceneDev& sc, int32_t t) {
    const float4* tp = sc.tris + 3 * (int64_t)t;
    TriRec r;
    r.a = tp[0];
    r.b = tp[1];
    r.c = tp[2];
    return r;
}
// Its geometric normal (triangle.cc:45-47).
__device__ inline v3f tri_normal(const TriRec& t) {
    return normalize(cross(xyz(t.b) - xyz(t.a), xyz(t.c) - xyz(t.a)));
}
// Its material.
__device__ inline int32_t tri_material(const TriRec& t) { return __float_as_int(t.b.w); }
__device__ inline int32_t tri_orig_id(const SceneDev& sc, int32_t t) {
    return __float_as_int(sc.tris[3 * (int64_t)t].w);
}
