// subsurface.hip -- the dipole diffusion sum of translucent surfaces on gfx950.
//
// Restates SubsurfaceIntegrator::irradiance (sources/subsurface_integrator.cc:
// 147-167, 234-238) with DipoleBSSRDF::operator() (sources/bssrdf.cc:92-104):
// for an eye path transmitted into a BSSRDF surface at x,
//   M_o(x) = sum_j R_d(|x - x_j|^2) E_j A_j,   L = (1 - F_dr) / pi * M_o,
// over all surface points j (the reference walks an octree cut of the same
// sum).  R_d per channel, with d+ = sqrt(d^2 + z+^2), d- = sqrt(d^2 + z-^2):
//   R_d = alpha' / (4 pi sigma_tr) (z+ (sigma_tr d+ + 1) e^{-sigma_tr d+} / d+^3
//                                   - z- (sigma_tr d- + 1) e^{-sigma_tr d-} / d-^3),
// clamped at 0, with the true exponential (the reference's Schraudolph
// approximation, sources/vector3d.cc:11-16, is not reproduced).
//
// N-body layout: a wave holds 64 eye hits in registers and walks a range of the
// points, staged through its own LDS in tiles of 128 (position and irradiance),
// every lane reading the tile from the same address (broadcast).  Sums in FP32:
// a plain partial sum per tile, Kahan-compensated across tiles, per channel.
// The bound is VALU issue, so what matters is that every SIMD has waves and
// that a pair costs few instructions:
// - hits and points are both split (dipole_split), so that a few hits fill the
//   chip too; the partial sums of a hit are added in order by k_dipole_sum;
// - lengths are in units of 1 / (sigma_tr log2 e) (DipoleDev), where a source
//   takes 6 full-rate and 2 transcendental instructions in place of 8 and 2
//   (a pair: 51 and 12).  Materials whose constants leave FP32's middle range
//   take the plain form.
// A call with 12,345 hits x 60,007 points, one block per 256 hits before, takes
// 13.3 -> 1.57 ms (4.7e11 pairs/s, copies included), one with 100 x 60,000 11.9 ->
// 0.31 ms; the error against 64 bits is 5.7e-8 against 6.4e-8 there (shorter
// tiles, fewer roundings).
#include "internal.h"

namespace {

struct Kahan3 {
    float s[3] = {0.0f, 0.0f, 0.0f};
    float c[3] = {0.0f, 0.0f, 0.0f};
    __device__ __forceinline__ void add(int k, float v) {
        const float y = v - c[k];
        const float t = s[k] + y;
        c[k] = (t - s[k]) - y;
        s[k] = t;
    }
};

// Per-hit constants of one channel: z+^2, z-^2, sigma_tr log2(e) for exp2,
// z sigma_tr and z for the (sigma_tr d + 1) z factors, alpha' / (4 pi sigma_tr)
struct DipolePlain {
    float zp2[3], zn2[3], trl[3], ztp[3], zp[3], ztn[3], zn[3], k[3];
    __device__ __forceinline__ explicit DipolePlain(const DipoleDev& D) {
        const float log2e = 1.4426950408889634f;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            zp2[c] = D.zp[c] * D.zp[c];
            zn2[c] = D.zn[c] * D.zn[c];
            trl[c] = D.tr[c] * log2e;
            ztp[c] = D.zp[c] * D.tr[c];
            zp[c] = D.zp[c];
            ztn[c] = D.zn[c] * D.tr[c];
            zn[c] = D.zn[c];
            k[c] = D.k[c];
        }
    }
    // z (sigma_tr d + 1) e^{-sigma_tr d} / d^3 with d^2 = s (s >= z^2 > 0, so the
    // raw reciprocal square root and exp2 need no denormal handling)
    static __device__ __forceinline__ float source(float s, float trl, float zt, float z) {
        const float id = __builtin_amdgcn_rsqf(s);
        const float d = s * id;
        const float e = __builtin_amdgcn_exp2f(-trl * d);
        return __builtin_fmaf(zt, d, z) * e * (id * id * id);
    }
    __device__ __forceinline__ float profile(int c, float d2) const {
        const float r = source(d2 + zp2[c], trl[c], ztp[c], zp[c]) - source(d2 + zn2[c], trl[c], ztn[c], zn[c]);
        return fmaxf(k[c] * r, 0.0f);
    }
    __device__ __forceinline__ float weight(int) const { return 1.0f; }
};

// The same in lengths of 1 / (sigma_tr log2 e): see DipoleDev.
struct DipoleScaled {
    float scale[3], at_p[3], at_n[3], ratio[3], w[3];
    __device__ __forceinline__ explicit DipoleScaled(const DipoleDev& D) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            scale[c] = D.scale[c];
            at_p[c] = D.at_p[c];
            at_n[c] = D.at_n[c];
            ratio[c] = D.ratio[c];
            w[c] = D.weight[c];
        }
    }
    static __device__ __forceinline__ float source(float s) {
        const float id = __builtin_amdgcn_rsqf(s);
        const float e = __builtin_amdgcn_exp2f(-(s * id));
        return (id + 0.693147180559945309f) * (id * id) * e;
    }
    __device__ __forceinline__ float profile(int c, float d2) const {
        const float p = source(__builtin_fmaf(d2, scale[c], at_p[c]));
        const float n = source(__builtin_fmaf(d2, scale[c], at_n[c]));
        return fmaxf(__builtin_fmaf(-ratio[c], n, p), 0.0f);
    }
    __device__ __forceinline__ float weight(int c) const { return w[c]; }
};

// How n hits are split: groups of 64, and the ranges of tiles each takes.
struct DipoleSplit {
    int64_t n, groups, tiles;
    int64_t ranges;
};
__device__ __forceinline__ DipoleSplit dipole_split(const DipoleArgs& a) {
    DipoleSplit s;
    s.n = a.count_src ? (int64_t)a.count_src->sss_hits : a.n_hit;
    s.groups = (s.n + 63) / 64;
    s.tiles = (a.n_pts + DIPOLE_TILE - 1) / DIPOLE_TILE;
    s.ranges = s.groups > 0 ? max((int64_t)1, min(s.tiles, DIPOLE_UNITS / s.groups)) : 1;
    return s;
}

__device__ __forceinline__ void dipole_out(const DipoleArgs& a, int64_t i, float dip_out, const float sum[3]) {
    const float4 w = a.hit_w[i];
    const float f = dip_out * a.area;
    const float Lo[3] = {w.x * f * sum[0], w.y * f * sum[1], w.z * f * sum[2]};
    const int64_t pix = (int64_t)__float_as_uint(w.w);
    if (a.img_sum) {
        for (int c = 0; c < 3; c++) kahan_add(a.img_sum, a.img_comp, 3 * pix + c, Lo[c]);
    } else {
        for (int c = 0; c < 3; c++) a.out_rgb[3 * i + c] = Lo[c];
    }
}

// One wave per unit (64 hits, a range of tiles), in turns.
template <class Dipole>
__global__ __launch_bounds__(256) void k_dipole(DipoleArgs a) {
    __shared__ float4 s_pe[4][DIPOLE_TILE];  // position, red
    __shared__ float2 s_e[4][DIPOLE_TILE];   // green, blue
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const DipoleSplit sp = dipole_split(a);
    for (int64_t u = (int64_t)blockIdx.x * 4 + wave; u < sp.groups * sp.ranges; u += (int64_t)gridDim.x * 4) {
        const int64_t i = (u / sp.ranges) * 64 + lane;
        const int64_t range = u % sp.ranges;
        const bool active = i < sp.n;
        float4 hp = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (active) hp = a.hit_pos[i];
        const DipoleDev& D = a.dip[active ? __float_as_int(hp.w) : 0];
        const Dipole L(D);
        Kahan3 acc;
        const int64_t t1 = (range + 1) * sp.tiles / sp.ranges;
        for (int64_t t = range * sp.tiles / sp.ranges; t < t1; t++) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = lane; k < DIPOLE_TILE; k += 64) {
                const int64_t j = t * DIPOLE_TILE + k;
                float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                float2 e = make_float2(0.0f, 0.0f);
                if (j < a.n_pts) {
                    p = a.pts[j];
                    p.w = a.E[3 * j];
                    e = make_float2(a.E[3 * j + 1], a.E[3 * j + 2]);
                }
                s_pe[wave][k] = p;
                s_e[wave][k] = e;
            }
            // the tile is the wave's own: its LDS operations run in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            float part[3] = {0.0f, 0.0f, 0.0f};
            for (int k = 0; k < DIPOLE_TILE; k++) {
                const float4 p = s_pe[wave][k];
                const float2 e = s_e[wave][k];
                const float dx = hp.x - p.x, dy = hp.y - p.y, dz = hp.z - p.z;
                const float d2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
                part[0] = __builtin_fmaf(L.profile(0, d2), p.w, part[0]);
                part[1] = __builtin_fmaf(L.profile(1, d2), e.x, part[1]);
                part[2] = __builtin_fmaf(L.profile(2, d2), e.y, part[2]);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int c = 0; c < 3; c++) acc.add(c, part[c]);
        }
        if (!active) continue;
        if (sp.ranges > 1) {
            float* p = a.part + (range * sp.groups * 64 + i) * 6;
            for (int c = 0; c < 3; c++) {
                p[c] = acc.s[c] * L.weight(c);
                p[3 + c] = acc.c[c] * L.weight(c);
            }
        } else {
            float sum[3];
            for (int c = 0; c < 3; c++) sum[c] = acc.s[c] * L.weight(c);
            dipole_out(a, i, D.out, sum);
        }
    }
}

// The partial sums of a hit, in the order of their ranges.
__global__ __launch_bounds__(256) void k_dipole_sum(DipoleArgs a) {
    const DipoleSplit sp = dipole_split(a);
    if (sp.ranges <= 1) return;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < sp.n; i += (int64_t)gridDim.x * 256) {
        Kahan3 acc;
        for (int64_t r = 0; r < sp.ranges; r++) {
            const float* p = a.part + (r * sp.groups * 64 + i) * 6;
            for (int c = 0; c < 3; c++) {
                acc.add(c, p[c]);
                acc.add(c, -p[3 + c]);
            }
        }
        dipole_out(a, i, a.dip[__float_as_int(a.hit_pos[i].w)].out, acc.s);
    }
}

// Issue-rate probes: eight independent chains per lane so latency is hidden;
// one store per thread
#define PROBE_ITERS 4096
__global__ __launch_bounds__(256) void k_probe_fma(float* out, float a, float b) {
    float x[8];
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = (float)threadIdx.x * 1e-3f + (float)k;
    for (int i = 0; i < PROBE_ITERS; i++) {
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = __builtin_fmaf(x[k], a, b);
    }
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) s += x[k];
    out[(int64_t)blockIdx.x * 256 + threadIdx.x] = s;
}
__global__ __launch_bounds__(256) void k_probe_exp(float* out, float a, float b) {
    float x[8];
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = (float)threadIdx.x * 1e-6f + (float)k * 1e-3f;
    for (int i = 0; i < PROBE_ITERS; i++) {
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = __builtin_amdgcn_exp2f(x[k]) * a + b;
    }
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) s += x[k];
    out[(int64_t)blockIdx.x * 256 + threadIdx.x] = s;
}

}  // namespace

// wave instructions per launch: 8 chains x PROBE_ITERS per wave (FMA); the
// exp probe issues one v_exp_f32 and one v_fma_f32 per chain step
void launch_issue_probe(hipStream_t s, float* out, int blocks, int which) {
    if (which == 0) hipLaunchKernelGGL(k_probe_fma, dim3((unsigned)blocks), dim3(256), 0, s, out, 0.999f, 0.001f);
    else hipLaunchKernelGGL(k_probe_exp, dim3((unsigned)blocks), dim3(256), 0, s, out, 0.5f, 0.001f);
}
int64_t issue_probe_wave_instr(int which) { return (which == 0 ? 8 : 16) * (int64_t)PROBE_ITERS; }

void launch_dipole(hipStream_t s, const DipoleArgs& a) {
    if (a.n_hit <= 0 || a.n_pts <= 0) return;
    // a.n_hit bounds the hits; waves without a unit end at once
    const dim3 g((unsigned)std::min<int64_t>((dipole_units(a.n_hit, a.n_pts) + 3) / 4, DIPOLE_UNITS / 4));
    if (a.scaled) hipLaunchKernelGGL(k_dipole<DipoleScaled>, g, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(k_dipole<DipolePlain>, g, dim3(256), 0, s, a);
    if (dipole_part_words(a.n_hit, a.n_pts) > 0)
        hipLaunchKernelGGL(k_dipole_sum, dim3((unsigned)std::min<int64_t>((a.n_hit + 255) / 256, 4096)), dim3(256), 0, s, a);
}
