// rc_cascade.hip -- per-level interval march, top-down bilinear merge,
// 4-child direction reduction, and the level-0 gather to irradiance.
//
// None of this exists in the reference (its only pass is the forward raster,
// src/renderer.rs:559-613); the maths is Sannikov's radiance cascades (2023):
//
//   march  : from c = ((px+1/2)s, (py+1/2)s) along theta_k, t from t0: sample
//            q = floor(c + t dir) (fused multiply-add per axis); off-image ->
//            (0, alpha 1); SDF(q) < 1/2 -> (E(q), alpha 0); else
//            t += max(SDF(q), 1); t >= t1 -> (0, alpha 1).
//   merge  : R_i(p,k) = march + alpha * bilinear_b A_{i+1}(b, k) over the 4
//            upper probes around p (upper coordinate p/2 - 1/4, indices
//            clamped, weights 3/4 and 1/4: x first, then y).
//   reduce : A_i(p,k') = 1/4 ((R(4k') + R(4k'+1)) + (R(4k'+2) + R(4k'+3))),
//            the only form in which level i-1 reads level i.
//   gather : irradiance(pixel) = bilinear over the level-0 fluence A_0.
//
// Work mapping of a level that marches its own rays (a level marched before by
// k_march_all is merged by k_merge): a workgroup (4 wave64) owns TX x TY probes x KD consecutive
// directions, lanes direction-fastest.  The 4 children of a level-(i-1)
// direction sit in one lane quad, so the reduction is two DPP quad
// permutations and no LDS.  Before marching, the workgroup stages the upper
// level's probe neighbourhood for its direction slice in LDS (one global read
// per texel instead of 16 L2 reads per ray).  Rays that hit skip the merge.
#include <algorithm>

#include "rc_internal.hpp"
#include "rc_march.hpp"

namespace rc {

// One ray with SPEC-deep speculation.  After a sample with distance d the
// next sample is exactly t + max(d, 1); a ray grazing a surface keeps taking
// the same step, so each round also loads the SPEC-1 samples that follow if
// the step stays unchanged (positions built with the same fp32 additions the
// sequential march would make).  The samples are then checked in order; the
// run of accepted ones ends at the first sample whose step differs, which
// starts the next round.  The visited sample sequence, and so every result
// bit, is that of the one-sample-per-step march.
struct Ray {
    float cx, cy, dx, dy, t, guess;
    int code;
    bool alive;
};

__device__ inline Ray ray_begin(float cx, float cy, float dx, float dy, float t0, float t1, bool active)
{
    return Ray{cx, cy, dx, dy, t0, 1.0f, kRayT1, active && t0 < t1};
}

template <int SPEC>
__device__ inline void ray_round(Ray &r, const SdfField &f, float t1)
{
    float p[SPEC];
    int ix[SPEC], iy[SPEC];
    uint32_t c[SPEC];
    p[0] = r.t;
#pragma unroll
    for (int j = 1; j < SPEC; ++j) p[j] = p[j - 1] + r.guess;
#pragma unroll
    for (int j = 0; j < SPEC; ++j) {
        ix[j] = floor_i32(fmaf(p[j], r.dx, r.cx));
        iy[j] = floor_i32(fmaf(p[j], r.dy, r.cy));
        c[j] = sdf_code(f, ix[j], iy[j]);
    }
    bool go = true;
#pragma unroll
    for (int j = 0; j < SPEC; ++j) {
        if (!go) continue;
        if (j > 0 && !(p[j] < t1)) {  // the previous step reached the interval end
            r.alive = false;
            go = false;
            continue;
        }
        if (c[j] == 0) {
            const bool ins = (uint32_t)ix[j] < (uint32_t)f.W && (uint32_t)iy[j] < (uint32_t)f.H;
            r.code = ins ? pixel_index(ix[j], iy[j], f.W) : kRayExit;
            r.alive = false;
            go = false;
            continue;
        }
        const float step = step_of_code(c[j]);
        if (j + 1 < SPEC && step == r.guess) continue;  // p[j+1] == p[j] + step
        r.t = p[j] + step;
        r.guess = step;
        r.alive = r.t < t1;
        go = false;
    }
}

// Level i >= 1.  Workgroup tile: TX x (TY*RPT) probes x KD directions; lane
// (probe column, direction) owns the RPT probes stacked TY rows apart.
template <int TX, int TY, int KD, int RPT, Storage S, bool UPPER, bool FROM_CODES>
__device__ __forceinline__ void level_body(const LevelArgs &a, int lb)
{
    static_assert(TX * TY * KD == kBlock, "a tile row block holds 256 rays");
    using TT = Texel<S>;
    constexpr int TYR = TY * RPT;
    constexpr int UCX = TX / 2 + 2, UCY = TYR / 2 + 2;
    __shared__ float4 su[UPPER ? UCX * UCY * KD : 1];

    const int tiles_x = (a.PX + TX - 1) / TX;
    const int slices = a.N / KD;
    const int slice = lb % slices, tile = lb / slices;
    const int px0 = (tile % tiles_x) * TX, py0 = (tile / tiles_x) * TYR, k0 = slice * KD;

    const int kk = threadIdx.x % KD, pl = threadIdx.x / KD;
    const int px = px0 + pl % TX, pyb = py0 + pl / TX, k = k0 + kk;

    // 32-bit indices: a level holds fewer than 2^32 rays (W, H <= 16384), N
    // is a power of two, and probe rows and columns are below 2^24
    const int log2n = 31 - __builtin_clz(a.N);
    const int ulx = (px0 - 1) >> 1, uly = (py0 - 1) >> 1;
    const uint32_t plane = __umul24((uint32_t)a.W, (uint32_t)a.H);
    bool active[RPT];
    int hitq[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j) active[j] = px < a.PX && pyb + j * TY < a.PY;

    // The upper level's neighbourhood for this direction slice, staged in
    // LDS: UN texels per thread, loaded to registers first.
    constexpr int UTOT = UCX * UCY * KD, UN = UPPER ? (UTOT + kBlock - 1) / kBlock : 0;
    typename TT::T ureg[UN > 0 ? UN : 1];
    auto stage_loads = [&]() {
        const typename TT::T *up = (const typename TT::T *)a.upper;
#pragma unroll
        for (int n = 0; n < UN; ++n) {
            const int i = (int)threadIdx.x + n * kBlock;
            if (i < UTOT) {
                const int j = i % KD, sx = (i / KD) % UCX, sy = i / (KD * UCX);
                const int ux = min(max(ulx + sx, 0), a.UX - 1), uy = min(max(uly + sy, 0), a.UY - 1);
                ureg[n] = up[((__umul24((uint32_t)uy, (uint32_t)a.UX) + (uint32_t)ux) << log2n) + (uint32_t)(k0 + j)];
            }
        }
    };
    auto stage_stores = [&]() {
#pragma unroll
        for (int n = 0; n < UN; ++n) {
            const int i = (int)threadIdx.x + n * kBlock;
            if (i < UTOT) su[i] = TT::unpack(ureg[n]);
        }
        __syncthreads();
    };
    // the emission of each ray's hit pixel (rgb; zero for a miss)
    float3 ev[RPT];
    auto gather_hits = [&]() {
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            ev[j] = make_float3(0.f, 0.f, 0.f);
            if (active[j] && hitq[j] >= 0) {
                const uint32_t q = (uint32_t)hitq[j];
                if (a.emis4) {
                    const float4 e = a.emis4[emis_index_of(q, a.W, emis_rcp(a.W))];
                    ev[j] = make_float3(e.x, e.y, e.z);
                } else {
                    ev[j] = make_float3(a.emissive[q], a.emissive[plane + q], a.emissive[2 * plane + q]);
                }
            }
        }
    };

    if (FROM_CODES) {
        // the rays were marched by the split march, which did not merge this,
        // the top level
        static_assert(!UPPER || !FROM_CODES, "a level with an upper one is merged from codes by merge_body");
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int py = min(pyb + j * TY, a.PY - 1);
            hitq[j] = a.codes[((__umul24((uint32_t)py, (uint32_t)a.PX) + (uint32_t)min(px, a.PX - 1)) << log2n) +
                              (uint32_t)k];
        }
        gather_hits();
    } else {
        if (UPPER) {
            stage_loads();
            stage_stores();
        }
        const float2 dir = a.dirs[k];
        float cx[RPT], cy[RPT];
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int py = pyb + j * TY;
            cx[j] = ((float)px + 0.5f) * a.spacing;
            cy[j] = ((float)py + 0.5f) * a.spacing;
        }
        march_rays<RPT>(sdf_field(a.sdf, a.W, a.H), cx, cy, dir.x, dir.y, a.t0, a.t1, active, hitq);
        if (a.dbg_codes) {
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int py = pyb + j * TY;
                if (active[j])
                    a.dbg_codes[((__umul24((uint32_t)py, (uint32_t)a.PX) + (uint32_t)px) << log2n) + (uint32_t)k] =
                        hitq[j];
            }
        }
        gather_hits();
    }

#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int py = pyb + j * TY;
        float r = 0.f, g = 0.f, b = 0.f, al = 0.f;
        if (active[j]) {
            if (hitq[j] >= 0) {
                r = ev[j].x;
                g = ev[j].y;
                b = ev[j].z;
            } else {
                al = 1.0f;
                if (UPPER) {
                    const int sx = ((px - 1) >> 1) - ulx, sy = ((py - 1) >> 1) - uly;
                    const float4 u00 = su[(sy * UCX + sx) * KD + kk];
                    const float4 u10 = su[(sy * UCX + sx + 1) * KD + kk];
                    const float4 u01 = su[((sy + 1) * UCX + sx) * KD + kk];
                    const float4 u11 = su[((sy + 1) * UCX + sx + 1) * KD + kk];
                    const float3 v = bilerp4(u00, u10, u01, u11, px, py);
                    r = v.x;
                    g = v.y;
                    b = v.z;
                }
            }
        }
        r = quad_sum(r) * 0.25f;
        g = quad_sum(g) * 0.25f;
        b = quad_sum(b) * 0.25f;
        al = quad_sum(al) * 0.25f;
        if (active[j] && (kk & 3) == 0) {
            typename TT::T *out = (typename TT::T *)a.out;
            out[((__umul24((uint32_t)py, (uint32_t)a.PX) + (uint32_t)px) << (log2n - 2)) + (uint32_t)(k >> 2)] =
                TT::pack(make_float4(r, g, b, al));
        }
    }
}

template <int TX, int TY, int KD, int RPT, Storage S, bool UPPER, bool FROM_CODES>
__global__ __launch_bounds__(kBlock) void k_level(LevelArgs a)
{
    level_body<TX, TY, KD, RPT, S, UPPER, FROM_CODES>(a, xcd_band(blockIdx.x, gridDim.x));
}

// The merge of level i from its pre-marched codes, 1 <= i < L - 1.  A lane owns
// one direction of a 2x2 block of probes (even column and row first), so the
// four bilinear footprints are 3x3 upper texels, their weights are constants
// and the footprints' x interpolations are shared by two rows of probes; the
// texels are read straight from memory, 64 (or 16) consecutive directions a
// wave, without LDS or a barrier.  A quad of lanes holds the 4 children of the
// 4 probes' next-lower direction: two exchanges leave lane q with probe q's sum
// in the order (v0 + v1) + (v2 + v3), and every lane stores one texel.
// Bound by latency and the hits' gathers: 24 us for the 4 merges of a
// 1920x1080 frame where a fifth of the pixels emit, 32 to 36 where more do (28
// and 40 with the emission row by row), 45 in the staged form of level_body
// (190 VALU per 128 rays, here 215 to 235 per 256 and 56 more in a wave with a
// hit), 63 and 184 at 3840x2160 in half storage.
__device__ inline float quad_exchange(float keep, float send, int ctrl_xor)
{
    const int o = ctrl_xor == 1 ? __builtin_amdgcn_mov_dpp(__float_as_int(send), 0xB1, 0xF, 0xF, false)
                                : __builtin_amdgcn_mov_dpp(__float_as_int(send), 0x4E, 0xF, 0xF, false);
    return keep + __int_as_float(o);
}

// Workgroups of 4 waves: 4x4 probes x 64 directions, or 8x8 probes x 16 (level 1).
// GATED: the tile fallback's, nothing when no tile is flagged and only the
// probes the flagged tiles need.
template <Storage S, bool NARROW, bool GATED>
__device__ __forceinline__ void merge_body(const LevelArgs &a, int lb)
{
    using TT = Texel<S>;
    if (GATED && *a.gate == 0) return;
    const int log2n = 31 - __builtin_clz(a.N);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int BX = (a.PX + 1) >> 1, BY = (a.PY + 1) >> 1;
    int bx, by, k;
    if (NARROW) {
        const int gx = (BX + 3) >> 2;
        bx = (lb % gx) * 4 + (lane >> 4);
        by = (lb / gx) * 4 + wave;
        k = lane & 15;
    } else {
        const int slices = a.N >> 6, gx = (BX + 1) >> 1;
        const int tile = lb / slices;
        bx = (tile % gx) * 2 + (wave & 1);
        by = (tile / gx) * 2 + (wave >> 1);
        k = (lb % slices) * 64 + lane;
    }
    const int qx = lane & 1, qy = (lane >> 1) & 1;  // the probe whose sum this lane ends with
    if (by >= BY) return;                           // wave-uniform
    if (!NARROW && bx >= BX) return;
    bool store = 2 * bx + qx < a.PX && 2 * by + qy < a.PY;
    if (GATED) {
        store = store && a.need[(2 * by + qy) * a.PX + 2 * bx + qx] != 0;
        if (!__any(store)) return;
    }

    uint32_t ux[3], uy[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        ux[j] = (uint32_t)min(max(bx - 1 + j, 0), a.UX - 1);
        uy[j] = __umul24((uint32_t)min(max(by - 1 + j, 0), a.UY - 1), (uint32_t)a.UX);
    }
    const typename TT::T *up = (const typename TT::T *)a.upper;
    int code[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t px = (uint32_t)min(2 * bx + (q & 1), a.PX - 1), py = (uint32_t)min(2 * by + (q >> 1), a.PY - 1);
        code[q] = a.codes[((__umul24(py, (uint32_t)a.PX) + px) << log2n) + (uint32_t)k];
        // the gated march left the other probes' codes as they were
        if (GATED && a.need[py * a.PX + px] == 0) code[q] = kRayExit;
    }
    typename TT::T raw[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) raw[r][c] = up[((uy[r] + ux[c]) << log2n) + (uint32_t)k];
    // hits take their pixel's emission: the 4 loads in one batch (a miss reads
    // pixel 0's) in a wave with a hit; each under its own lanes' mask, they wait
    // for one another
    float4 e[4] = {};
    if (__any(max(max(code[0], code[1]), max(code[2], code[3])) >= 0)) {
        const float rcp = emis_rcp(a.W);
#pragma unroll
        for (int q = 0; q < 4; ++q) e[q] = a.emis4[emis_index_of((uint32_t)max(code[q], 0), a.W, rcp)];
    }
    float v[4][4];
    // x interpolation of the 3 rows at the even and the odd column
    float x[3][2][3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const float4 u0 = TT::unpack(raw[r][0]), u1 = TT::unpack(raw[r][1]), u2 = TT::unpack(raw[r][2]);
        x[r][0][0] = fmaf(0.75f, u1.x, 0.25f * u0.x);
        x[r][0][1] = fmaf(0.75f, u1.y, 0.25f * u0.y);
        x[r][0][2] = fmaf(0.75f, u1.z, 0.25f * u0.z);
        x[r][1][0] = fmaf(0.25f, u2.x, 0.75f * u1.x);
        x[r][1][1] = fmaf(0.25f, u2.y, 0.75f * u1.y);
        x[r][1][2] = fmaf(0.25f, u2.z, 0.75f * u1.z);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int dx = q & 1, dy = q >> 1;
        const float w1 = dy ? 0.25f : 0.75f, w0 = 1.0f - w1;
        const bool hit = code[q] >= 0;
        const float4 h = e[q];
        v[q][0] = hit ? h.x : fmaf(w1, x[dy + 1][dx][0], w0 * x[dy][dx][0]);
        v[q][1] = hit ? h.y : fmaf(w1, x[dy + 1][dx][1], w0 * x[dy][dx][1]);
        v[q][2] = hit ? h.z : fmaf(w1, x[dy + 1][dx][2], w0 * x[dy][dx][2]);
        v[q][3] = hit ? 0.0f : 1.0f;
    }
    float s[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float lo = quad_exchange(qx ? v[1][c] : v[0][c], qx ? v[0][c] : v[1][c], 1);
        const float hi = quad_exchange(qx ? v[3][c] : v[2][c], qx ? v[2][c] : v[3][c], 1);
        s[c] = quad_exchange(qy ? hi : lo, qy ? lo : hi, 2) * 0.25f;
    }
    if (store) {
        const uint32_t p = __umul24((uint32_t)(2 * by + qy), (uint32_t)a.PX) + (uint32_t)(2 * bx + qx);
        ((typename TT::T *)a.out)[(p << (log2n - 2)) + (uint32_t)(k >> 2)] = TT::pack(make_float4(s[0], s[1], s[2], s[3]));
    }
}

template <Storage S, bool NARROW, bool GATED>
__global__ __launch_bounds__(kBlock) void k_merge(LevelArgs a)
{
    merge_body<S, NARROW, GATED>(a, xcd_band(blockIdx.x, gridDim.x));
}

int merge_blocks(int PX, int PY, int N)
{
    const int BX = (PX + 1) >> 1, BY = (PY + 1) >> 1;
    return N < 64 ? ((BX + 3) >> 2) * ((BY + 3) >> 2) : ((BX + 1) >> 1) * ((BY + 1) >> 1) * (N >> 6);
}

// One level over a work list of views (each job a view's LevelArgs; the top
// level of a view has no upper level, so UPPER is taken per job).
template <int TX, int TY, int KD, int RPT, Storage S, bool FROM_CODES>
__global__ __launch_bounds__(kBlock) void k_level_batch(const LevelArgs *__restrict__ jobs,
                                                        const int *__restrict__ begins, int njobs)
{
    const int b = xcd_band(blockIdx.x, gridDim.x);
    const int j = batch_job(begins, njobs, b);
    const LevelArgs a = jobs[j];
    const int lb = b - begins[j];
    if (!a.upper) level_body<TX, TY, KD, RPT, S, false, FROM_CODES>(a, lb);
    else if constexpr (!FROM_CODES) level_body<TX, TY, KD, RPT, S, true, false>(a, lb);
    else if (a.N < 64) merge_body<S, true, false>(a, lb);
    else merge_body<S, false, false>(a, lb);
}

// Level 0 (4 directions, interval [0,2)) fused with the gather.  A tile owns
// 16x12 level-0 probes = 32x24 pixels (each output row one 128-byte line); a
// thread marches one probe of the tile plus its 1-probe halo (18x14 = 252
// probes, the pixels' bilinear footprint), all 4 directions at once, and
// writes the probe's fluence to LDS; the pixels then read it bilinearly and
// write planar fp32 irradiance.
//
// Every direction of a probe starts at the probe centre (t = 0), so the first
// sample is shared.  Distances are whole pixels below 128, hence a first
// value of 0 is a hit for all 4 rays, a value >= 2 ends all 4 intervals, and
// only a value of exactly 1 takes a second, per-direction sample at t = 1,
// after which every ray has ended (1 + max(d, 1) >= 2).  These are the steps
// the generic interval march takes, so the codes are the same; the fluence
// is the same sum ((v0 + v1) + (v2 + v3)) / 4 of the per-direction values.
template <Storage S, bool UPPER>
__device__ __forceinline__ void level0_body(const LevelArgs &a, float *__restrict__ irr, float *__restrict__ dbg,
                                            int lb)
{
    using TT = Texel<S>;
    constexpr int TX = kL0TX, TY = kL0TY, NX = TX + 2, NY = TY + 2, UCX = TX / 2 + 2, UCY = TY / 2 + 2;
    static_assert(NX * NY <= kBlock, "one probe per thread");
    __shared__ float4 su[UPPER ? UCX * UCY * 4 : 1];
    __shared__ float4 fl[NX * NY];

    const int tiles_x = (a.PX + TX - 1) / TX;
    const int px0 = (lb % tiles_x) * TX, py0 = (lb / tiles_x) * TY;
    const int ulx = (px0 - 2) >> 1, uly = (py0 - 2) >> 1;
    // 32-bit indices (W, H <= 16384: three planes hold fewer than 2^32 floats)
    const uint32_t plane = __umul24((uint32_t)a.W, (uint32_t)a.H);
    const int slot = threadIdx.x;
    const int sx = slot % NX, sy = slot / NX;
    const int px = px0 - 1 + sx, py = py0 - 1 + sy;
    const bool probe = slot < NX * NY && px >= 0 && py >= 0 && px < a.PX && py < a.PY;
    const SdfField sdf = sdf_field(a.sdf, a.W, a.H);
    const float cx = ((float)px + 0.5f) * 2.0f, cy = ((float)py + 0.5f) * 2.0f;
    const int ix = 2 * px + 1, iy = 2 * py + 1;  // floor of the probe centre (exact)
    const bool in0 = probe && (uint32_t)ix < (uint32_t)a.W && (uint32_t)iy < (uint32_t)a.H;
    // the first distance sample is issued before the upper level's loads, so
    // the march does not wait for them; they land in LDS after the march
    const float d0 = in0 ? sdf_value(sdf_code(sdf, ix, iy)) : 0.0f;
    // the emission of the first sample's pixel (the usual hit) in the same wave
    // of loads, so a hit there needs no dependent load
    const int q0 = in0 ? pixel_index(ix, iy, a.W) : 0;
    float ep0 = 0.f, ep1 = 0.f, ep2 = 0.f;
    if (in0) {
        ep0 = a.emissive[q0];
        ep1 = a.emissive[plane + q0];
        ep2 = a.emissive[2 * plane + q0];
    }
    constexpr int UN = UPPER ? (UCX * UCY * 4 + kBlock - 1) / kBlock : 1;
    typename TT::T ureg[UN];
    if (UPPER) {
        const typename TT::T *up = (const typename TT::T *)a.upper;
#pragma unroll
        for (int n = 0; n < UN; ++n) {
            const int i = threadIdx.x + n * kBlock;
            if (i < UCX * UCY * 4) {
                const int j = i & 3, ux0 = (i >> 2) % UCX, uy0 = (i >> 2) / UCX;
                const int ux = min(max(ulx + ux0, 0), a.UX - 1), uy = min(max(uly + uy0, 0), a.UY - 1);
                ureg[n] = up[((__umul24((uint32_t)uy, (uint32_t)a.UX) + (uint32_t)ux) << 2) + (uint32_t)j];
            }
        }
    }

    int code[4] = {kRayT1, kRayT1, kRayT1, kRayT1};
    if (probe) {
        if (!in0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) code[k] = kRayExit;
        } else if (d0 < 0.5f) {
#pragma unroll
            for (int k = 0; k < 4; ++k) code[k] = q0;
        } else if (march_step(d0) < 2.0f) {
            const float t = march_step(d0);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float2 dir = a.dirs[k];
                const int jx = floor_i32(fmaf(t, dir.x, cx)), jy = floor_i32(fmaf(t, dir.y, cy));
                if (!((uint32_t)jx < (uint32_t)a.W && (uint32_t)jy < (uint32_t)a.H)) {
                    code[k] = kRayExit;
                } else if (sdf_code(sdf, jx, jy) == 0) {
                    code[k] = pixel_index(jx, jy, a.W);
                }
            }
        }
    }
    if (a.dbg_codes && probe && sx >= 1 && sx <= TX && sy >= 1 && sy <= TY) {
#pragma unroll
        for (int k = 0; k < 4; ++k) a.dbg_codes[((size_t)py * a.PX + px) * 4 + k] = code[k];
    }
    float r[4], g[4], b[4], al[4];
    const bool one_hit = code[0] >= 0 && code[0] == code[1] && code[0] == code[2] && code[0] == code[3];
    if (one_hit) {
        // one hit pixel for all 4 directions: its emission once (already
        // loaded when it is the first sample's pixel)
        const bool first = code[0] == q0;
        const uint32_t c0 = (uint32_t)code[0];
        const float e0 = first ? ep0 : a.emissive[c0];
        const float e1 = first ? ep1 : a.emissive[plane + c0];
        const float e2 = first ? ep2 : a.emissive[2 * plane + c0];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            r[k] = e0;
            g[k] = e1;
            b[k] = e2;
            al[k] = 0.f;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            r[k] = g[k] = b[k] = 0.f;
            al[k] = code[k] >= 0 ? 0.f : 1.0f;
            if (code[k] >= 0) {
                const bool first = code[k] == q0;
                const uint32_t ck = (uint32_t)code[k];
                r[k] = first ? ep0 : a.emissive[ck];
                g[k] = first ? ep1 : a.emissive[plane + ck];
                b[k] = first ? ep2 : a.emissive[2 * plane + ck];
            }
        }
    }
    if (UPPER) {
#pragma unroll
        for (int n = 0; n < UN; ++n) {
            const int i = threadIdx.x + n * kBlock;
            // direction-major (su[k][y][x]): neighbouring probes read
            // neighbouring texels, so the merge's LDS reads do not conflict
            if (i < UCX * UCY * 4) su[(i & 3) * (UCX * UCY) + (i >> 2)] = TT::unpack(ureg[n]);
        }
        __syncthreads();
        if (probe && !one_hit) {
            const int usx = ((px - 1) >> 1) - ulx, usy = ((py - 1) >> 1) - uly;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (code[k] < 0) {
                    const float4 *sk = su + k * (UCX * UCY) + usy * UCX + usx;
                    const float4 u00 = sk[0], u10 = sk[1], u01 = sk[UCX], u11 = sk[UCX + 1];
                    const float3 v = bilerp4(u00, u10, u01, u11, px, py);
                    r[k] = v.x;
                    g[k] = v.y;
                    b[k] = v.z;
                }
            }
        }
    }
    if (probe) {
        const float4 f = make_float4(((r[0] + r[1]) + (r[2] + r[3])) * 0.25f, ((g[0] + g[1]) + (g[2] + g[3])) * 0.25f,
                                     ((b[0] + b[1]) + (b[2] + b[3])) * 0.25f,
                                     ((al[0] + al[1]) + (al[2] + al[3])) * 0.25f);
        fl[slot] = f;
        if (dbg && sx >= 1 && sx <= TX && sy >= 1 && sy <= TY) reinterpret_cast<float4 *>(dbg)[(size_t)py * a.PX + px] = f;
    }
    __syncthreads();

    // Pixels in 2x2 quads: pixel x = 2m interpolates probes m-1, m and x =
    // 2m+1 probes m, m+1 (indices clamped to the grid; the same in y), so a
    // quad reads 3x3 fluence texels for its 4 pixels, and with W even (and an
    // 8-byte aligned output) each row of it is one 8-byte store per plane.
    static_assert(TX * TY <= kBlock, "one quad per lane");
    if ((int)threadIdx.x < TX * TY) {
        const int m = px0 + (int)threadIdx.x % TX, n = py0 + (int)threadIdx.x / TX;
        const int x = 2 * m, y = 2 * n;
        if (x < a.W && y < a.H) {
            int cx[3], cy[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                cx[d] = min(max(m - 1 + d, 0), a.PX - 1) - (px0 - 1);
                cy[d] = min(max(n - 1 + d, 0), a.PY - 1) - (py0 - 1);
            }
            float4 f[3][3];
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) f[r][c] = fl[cy[r] * NX + cx[c]];
            float3 v[2][2];
#pragma unroll
            for (int dy = 0; dy < 2; ++dy)
#pragma unroll
                for (int dx = 0; dx < 2; ++dx)
                    v[dy][dx] = bilerp4(f[dy][dx], f[dy][dx + 1], f[dy + 1][dx], f[dy + 1][dx + 1], x + dx, y + dy);
            const bool x1 = x + 1 < a.W;
            const bool pair = x1 && (a.W & 1) == 0 && (reinterpret_cast<uintptr_t>(irr) & 7) == 0;
#pragma unroll
            for (int dy = 0; dy < 2; ++dy) {
                if (y + dy >= a.H) break;
                const uint32_t p = __umul24((uint32_t)(y + dy), (uint32_t)a.W) + (uint32_t)x;
                if (pair) {
                    *reinterpret_cast<float2 *>(irr + p) = make_float2(v[dy][0].x, v[dy][1].x);
                    *reinterpret_cast<float2 *>(irr + plane + p) = make_float2(v[dy][0].y, v[dy][1].y);
                    *reinterpret_cast<float2 *>(irr + 2 * plane + p) = make_float2(v[dy][0].z, v[dy][1].z);
                } else {
                    irr[p] = v[dy][0].x;
                    irr[plane + p] = v[dy][0].y;
                    irr[2 * plane + p] = v[dy][0].z;
                    if (x1) {
                        irr[p + 1] = v[dy][1].x;
                        irr[plane + p + 1] = v[dy][1].y;
                        irr[2 * plane + p + 1] = v[dy][1].z;
                    }
                }
            }
        }
    }
}

template <Storage S, bool UPPER>
__global__ __launch_bounds__(kBlock) void k_level0(LevelArgs a, float *__restrict__ irr, float *__restrict__ dbg)
{
    level0_body<S, UPPER>(a, irr, dbg, xcd_band(blockIdx.x, gridDim.x));
}

template <Storage S>
__global__ __launch_bounds__(kBlock) void k_level0_batch(const Level0Job *__restrict__ jobs,
                                                         const int *__restrict__ begins, int njobs)
{
    const int b = xcd_band(blockIdx.x, gridDim.x);
    const int j = batch_job(begins, njobs, b);
    const LevelArgs a = jobs[j].a;
    float *irr = jobs[j].irr;
    const int lb = b - begins[j];
    if (a.upper) level0_body<S, true>(a, irr, nullptr, lb);
    else level0_body<S, false>(a, irr, nullptr, lb);
}

// Canonical ray r = (py*PX + px)*N + k -> (px, py, k): the direction is the
// low log2(N) bits; probe / PX by an fp32 reciprocal, corrected to the exact
// quotient (probe < 2^24, so the estimate is off by at most one).
__device__ inline void decode_ray(const MarchLevel &L, int ray, int &px, int &py, int &k)
{
    k = ray & (L.N - 1);
    const int probe = ray >> L.log2n;
    py = (int)((float)probe * L.inv_px);
    px = probe - py * L.PX;
    if (px < 0) { --py; px += L.PX; }
    else if (px >= L.PX) { ++py; px -= L.PX; }
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// The order of a level's rays over the split march's slots.  Wave tiles: slot =
// T*64 + lane, T = (tile row * ntx + tile column) * slices + slice, lane =
// (probe in the tile, direction in the slice) with the direction fastest.  Rays
// with nearby start points and directions share a wave, so their march lengths
// are alike.  Canonical order is the wave tile of one probe x 64 directions,
// or, for level 1's 16 directions (wrap), the canonical index itself: 4
// consecutive probes, which may wrap to the next row.
// A packet T is one tile (row, column, slice) and lane constants: start points
// and addresses are a part of T's, scalar where a wave takes one packet at a
// time, plus a lane's, and the level's fields stay in scalar registers (read
// from the arguments per packet, one after another, they took a launch without
// march and stores to 14.7 us at 1920x1080).  Both forms of the split launch
// and the readback of its order place rays by this (where a lane takes several
// rays, T differs between lanes); the persistent form is canonical, by
// decode_ray.
struct RayOrder {
    int PX, PY, log2n, slots, tx_log, ty_log, ntx, rcp, kd_log, ns_log, smask;
    bool wrap;
    int lane, lk, lx, ly;
    uint32_t lat;  // the lane's part of its rays' canonical index
};
__device__ __forceinline__ RayOrder ray_order(const MarchLevel &L, int lane)
{
    RayOrder o;
    o.PX = uniform(L.PX), o.PY = uniform(L.PY), o.log2n = uniform(L.log2n), o.slots = uniform((int)L.slots);
    o.tx_log = uniform(L.tx_log), o.ty_log = uniform(L.ty_log);
    o.ntx = uniform(L.ntx), o.rcp = uniform((int)L.rcp_ntx);
    o.wrap = L.map == 0 && L.kd_log == 0;
    o.kd_log = uniform(o.wrap ? 4 : L.kd_log), o.ns_log = o.log2n - o.kd_log;
    o.smask = (1 << o.ns_log) - 1;
    o.lane = lane;
    o.lk = lane & ((1 << o.kd_log) - 1);
    const int pl = lane >> o.kd_log;
    o.lx = pl & ((1 << o.tx_log) - 1), o.ly = pl >> o.tx_log;
    o.lat = o.wrap ? (uint32_t)lane
                   : ((__umul24((uint32_t)o.ly, (uint32_t)o.PX) + (uint32_t)o.lx) << o.log2n) + (uint32_t)o.lk;
    return o;
}
// The lane's direction in packet T, as an offset into the level's table: the
// part of T's (lk is the lane's).
__device__ __forceinline__ int ray_slice(const RayOrder &o, int T) { return o.wrap ? 0 : (T & o.smask) << o.kd_log; }
// The probe of the lane's ray in packet T, and at: the part of T's of its
// canonical index (the other is lat).  False for a lane without a ray: past the
// last slot, or outside the probe grid in a ragged edge tile.  The quotient's
// estimate by the reciprocal is off by at most one either way.
__device__ __forceinline__ bool ray_place(const RayOrder &o, const MarchLevel &L, int T, int &px, int &py, uint32_t &at)
{
    if (o.wrap) {
        int k;
        const int ray = T * 64 + o.lane;
        const bool in = ray < o.slots;
        decode_ray(L, in ? ray : 0, px, py, k);
        at = (uint32_t)T * 64;
        return in;
    }
    const uint32_t tt = (uint32_t)T >> o.ns_log, ntx = (uint32_t)o.ntx;
    uint32_t ty = __umulhi(tt, (uint32_t)o.rcp);
    if (ty * ntx > tt) --ty;
    if (tt - ty * ntx >= ntx) ++ty;
    const int sx = (int)(tt - ty * ntx) << o.tx_log, sy = (int)ty << o.ty_log;
    px = sx + o.lx;
    py = sy + o.ly;
    at = ((uint32_t)(sy * o.PX + sx) << o.log2n) + (uint32_t)ray_slice(o, T);
    return px < o.PX && py < o.PY;
}
// The packets of wave `wave`: first, first + step, ... below end.  One ray a
// lane at a time: L.packets of them, L.stride apart, so that a group of L.stride
// waves shares L.stride * L.packets; M: the M next to each other.
struct Packets {
    int first, step, end;
};
__device__ __forceinline__ Packets wave_packets(const MarchLevel &L, int wave, int m)
{
    const int all = uniform((int)((L.slots + 63) >> 6));
    if (m == 1) {
        const int before = wave >> L.group_log << L.group_log;  // waves in the groups before this one's
        const int stride = uniform(L.stride), first = wave + before * (L.packets - 1);
        return Packets{first, stride, uniform(min(all, first + stride * L.packets))};
    }
    return Packets{wave * m, 1, min(wave * m + m, all)};
}

// All levels >= 1 marched by one launch; each ray's code (hit pixel, -1 left
// the image, -2 reached t1) is written in canonical order for the merge
// kernels.  The block list is level-major with the top level first, so the
// levels whose rays are longest start earliest, and the long dependent chains
// of different levels run concurrently instead of one kernel after another.
//
// With one ray a lane at a time (M = 1) see march_packets.  Otherwise a
// workgroup owns 64*M consecutive slots and lane l marches slots base+l,
// base+l+64, ... one after another without waiting for the other lanes: when
// its ray ends it starts the next one in the same loop iteration.
// Blocks go round-robin to the XCDs, which interleaves heavy and light tiles.
// A_top texel of a lane quad, merged in the march: the level kernel's
// arithmetic for a level without an upper level (quad sums of the 4 rays,
// times 1/4), stored by the quad's first lane.
__device__ inline void merge_top_quad(const MarchLevel &L, const float4 *__restrict__ emis4, int W, bool valid, int code,
                                      uint32_t at)
{
    float r = 0.f, g = 0.f, b = 0.f, al = 0.f;
    if (valid) {
        if (code >= 0) {
            const float4 e = emis4[emis_index_of((uint32_t)code, W, emis_rcp(W))];
            r = e.x;
            g = e.y;
            b = e.z;
        } else {
            al = 1.0f;
        }
    }
    r = quad_sum(r) * 0.25f;
    g = quad_sum(g) * 0.25f;
    b = quad_sum(b) * 0.25f;
    al = quad_sum(al) * 0.25f;
    if (valid && (at & 3) == 0) {
        const float4 v = make_float4(r, g, b, al);
        const uint32_t i = at >> 2;
        if (L.storage == (int)Storage::F32) ((float4 *)L.merged)[i] = v;
        else if (L.storage == (int)Storage::F16) ((uint2 *)L.merged)[i] = Texel<Storage::F16>::pack(v);
        else ((uint2 *)L.merged)[i] = Texel<Storage::BF16>::pack(v);
    }
}

// One round of a ray's march from t with SPEC samples: sample 0 at t and the
// next ones where the ray goes if the step stays `guess` (every t is a whole
// number below 2^24, so t + j guess is exact).  Sample j counts while the step
// of every one before it was the guess; the last that counts gives the next t
// and the next guess.  Branch-free, with the interval's end left to the caller:
// a sample beyond t1 can only leave t beyond t1.  Returns whether the ray goes
// on; otherwise t stopped at the sample that ended it (code 0: off-image or a
// hit), or at or past t1.  all: every sample's step was the guess.
template <int SPEC>
__device__ __forceinline__ bool march_round(const SdfField &f, float cx, float cy, float2 dir, float t1, float &t,
                                            float &guess, bool &all)
{
    float p[SPEC], step[SPEC];
    uint32_t c[SPEC];
    p[0] = t;
#pragma unroll
    for (int j = 1; j < SPEC; ++j) p[j] = p[j - 1] + guess;
#pragma unroll
    for (int j = 0; j < SPEC; ++j)
        c[j] = sdf_code(f, floor_i32(fmaf(p[j], dir.x, cx)), floor_i32(fmaf(p[j], dir.y, cy)));
#pragma unroll
    for (int j = 0; j < SPEC; ++j) step[j] = step_of_code(c[j]);
    float at = p[0], by = step[0];
    bool same = step[0] == guess;
#pragma unroll
    for (int j = 1; j < SPEC; ++j) {
        at = same ? p[j] : at;
        by = same ? step[j] : by;
        same = same && step[j] == guess;
    }
    all = same;
    t = at + by;
    guess = by;
    return by != 0.0f && t < t1;
}

// One ray per lane.  The median packet of 64 rays of a 1920x1080 frame ends
// after 1 to 2 samples and the longest ray takes 339 (791 at 3840x2160), so
// two things bounded a launch of one packet per wave: handing out 163,200
// one-wave workgroups takes 36 us alone (4.6 a ns), and a chain of 339
// dependent samples of 0.17 us each takes as long as the whole launch, 58 us.
// - A wave takes L.packets packets, L.stride apart, as a rule a grid's width of
//   waves (neighbouring packets hold rays of like length: 4 in a run gave one
//   wave 4 long ones, 66 us against 60), the next packet's directions read
//   while the present one marches.
// - A ray takes its first kMarchPlain samples one per step, in a branch-free
//   divergent loop on the raw byte code (lanes leave as their rays end), and
//   the rest kMarchTail at a time: 100 rounds instead of 339 samples for the
//   longest, in 2,500 of the packets.  Frames of 1920x1080 took 129.1, 128.4,
//   126.5 and 128.9 us with 8, 12, 16 and 24 plain samples, 151 with no others;
//   6 and 8 samples a round 126.3 and 128.5.
// - That pays where rays run along a surface and repeat their step.  Among
//   scattered pixels every step differs: a round takes one step for four
//   loads, and the loads bound the launch (1920x1080 with a thousandth of the
//   pixels lit: 587 us, 375 one sample a step).  So a wave first takes
//   kTailProbe rounds, and guesses on to the end of its rays if 1 in
//   kTailShare of them had all four steps alike; otherwise it takes kTailPlain
//   samples one per step, probes again, and waits twice as long each time.
//   (A launch too small to fill the chip, L.probe false, guesses always.)
//   That scene 373 us; 8 scenes of lit boxes 119.0 us on average, 118.3 guessing
//   always, and 6 to 20 us more where the choice is made anew every round: it
//   lies in the longest ray's chain.
// Both kinds of scene with the field's zeros outside the image.
constexpr int kMarchPlain = 16, kMarchTail = 4;
constexpr int kTailProbe = 2, kTailShare = 16, kTailPlain = 24;

template <int SPEC, bool GATED>
__device__ __forceinline__ void march_packets(const SdfField &field, const MarchLevel &L, int lb,
                                              const float4 *__restrict__ emis4)
{
    const int lane = (int)threadIdx.x & 63;
    SdfField f = field;
    f.W = uniform(f.W);
    f.H = uniform(f.H);
    f.skip = uniform(f.skip);
    const RayOrder o = ray_order(L, lane);
    const int spacing = uniform((int)L.spacing);
    const bool probe = L.probe;
    const float t0 = __int_as_float(uniform(__float_as_int(L.t0))), t1 = __int_as_float(uniform(__float_as_int(L.t1)));
    const float2 *dirs = L.dirs;
    int *codes = L.codes;
    const bool top = L.merged != nullptr;
    auto direction = [&](int T) -> float2 { return (dirs + ray_slice(o, T))[o.lk]; };

    const Packets p = wave_packets(L, lb, 1);
    float2 next = direction(p.first);
    for (int T = p.first; T < p.end; T += p.step) {
        const float2 dir = next;
        next = direction(T + p.step);
        int px, py;
        uint32_t at;
        bool valid = ray_place(o, L, T, px, py, at);
        if (GATED) {
            valid = valid && L.need[py * o.PX + px] != 0;
            if (!__any(valid)) continue;
        }
        // (p + 1/2) spacing, a whole number: spacing is even
        const float cx = (float)((int)__umul24((uint32_t)px, (uint32_t)spacing) + (spacing >> 1));
        const float cy = (float)((int)__umul24((uint32_t)py, (uint32_t)spacing) + (spacing >> 1));
        float t = t0;
        bool alive = valid && t < t1;
        float guess = 1.0f;
        if (SPEC == 1) {
            for (int step = 0; alive && step < kMarchPlain; ++step) {
                const uint32_t c = sdf_code(f, floor_i32(fmaf(t, dir.x, cx)), floor_i32(fmaf(t, dir.y, cy)));
                t = t + step_of_code(c);
                alive = c != 0 && t < t1;
            }
            if (alive) {
                int plain = kTailPlain;
                bool all;
                do {
                    if (probe) {
                        const int on = __popcll(__builtin_amdgcn_ballot_w64(true));
                        bool run = false;
#pragma unroll
                        for (int round = 0; round < kTailProbe; ++round) {
                            if (!alive) break;
                            alive = march_round<kMarchTail>(f, cx, cy, dir, t1, t, guess, all);
                            run = run || all;
                        }
                        if (__popcll(__builtin_amdgcn_ballot_w64(run)) * kTailShare < on) {
#pragma unroll 1
                            for (int step = 0; alive && step < plain; ++step) {
                                const uint32_t c = sdf_code(f, floor_i32(fmaf(t, dir.x, cx)), floor_i32(fmaf(t, dir.y, cy)));
                                guess = step_of_code(c);
                                t = t + guess;
                                alive = c != 0 && t < t1;
                            }
                            plain *= 2;  // a ray takes fewer than 2^16 samples (t1 < 2^16, steps of 1 at least)
                            continue;
                        }
                    }
                    while (alive) alive = march_round<kMarchTail>(f, cx, cy, dir, t1, t, guess, all);
                } while (alive);
            }
        } else {
            bool all;
            while (alive) alive = march_round<SPEC>(f, cx, cy, dir, t1, t, guess, all);
        }
        const int code = ray_code(f, t, t1, dir.x, dir.y, cx, cy);
        if (valid) (codes + at)[o.lat] = code;
        if (top) merge_top_quad(L, emis4, f.W, valid, code, at + o.lat);
    }
}

template <int SPEC, int M>
__device__ __forceinline__ void march_all_body(const uint8_t *sdf_codes, int W, int H, const MarchLevel &L, int lb,
                                               const float4 *__restrict__ emis4)
{
    const SdfField f = sdf_field(sdf_codes, W, H);
    if (M == 1) {
        march_packets<SPEC, false>(f, L, lb, emis4);
        return;
    }
    const RayOrder o = ray_order(L, (int)threadIdx.x);
    const Packets p = wave_packets(L, lb, M);

    int j = 0, T = p.first;
    bool valid = false;      // the slot holds a ray of the grid
    uint32_t at = 0;         // its canonical index (where its code goes)
    Ray r;
    auto start = [&]() {
        int px, py;
        valid = ray_place(o, L, T < p.end ? T : 0, px, py, at) && T < p.end;
        at += o.lat;
        const float2 dir = L.dirs[at & (uint32_t)(L.N - 1)];
        r = ray_begin(((float)px + 0.5f) * L.spacing, ((float)py + 0.5f) * L.spacing, dir.x, dir.y, L.t0, L.t1,
                      valid);
    };
    start();
    for (;;) {
        if (r.alive) ray_round<SPEC>(r, f, L.t1);
        if (j < M && !r.alive) {
            if (valid) L.codes[at] = r.code;
            T += p.step;
            if (++j < M) start();
        }
        if (!__any(j < M)) break;
    }
}

template <int SPEC, int M>
__global__ __launch_bounds__(kMarchBlock) void k_march_all(MarchAllArgs a)
{
    // the grid is (blocks of the largest level) x (levels): the level is
    // blockIdx.y, and workgroups are dispatched x-fastest, so the top level's
    // (longest) rays start first
    const MarchLevel &L = a.lev[blockIdx.y];
    if ((int)blockIdx.x >= L.blocks) return;
    march_all_body<SPEC, M>(a.sdf, a.W, a.H, L, (int)blockIdx.x, a.emis4);
}

// The tile fallback's split march: nothing when no tile is flagged, and only
// the probes the flagged tiles need.  A frame with no flagged tile pays for
// handing the workgroups out, so there are few: four waves each, and at most
// kGatedWaves waves a launch, which then take more packets.  Means of 4 scenes,
// in us, where the fallback marched level by level, with one wave a workgroup
// and no limit, and so:
//              no tile flagged       threshold 1         every tile
//   700x400     56.2  60.3  56.1   136.9  94.3  94.5   150.6  98.6  98.0
//   1366x768    79.0  83.1  76.9   201.1 127.3 128.3   255.7 148.2 148.9
//   1920x1080  102.2 110.8  96.8   269.0 169.3 169.2   335.3 205.7 211.3
//   3840x2160  283.9 278.0 261.8   742.7 511.4 514.7  1023.6 744.9 748.5
// (two waves, 32,768 at most: 57.7, 78.6, 97.4 and 261 unused, 99.0, 149.1,
// 209 and 742 with every tile; one wave, 32,768: 60.4, 82.9, 102.7 and 264
// unused.)
__global__ __launch_bounds__(kGatedBlock) void k_march_gated(MarchAllArgs a)
{
    const MarchLevel &L = a.lev[blockIdx.y];
    const int wave = (int)blockIdx.x * (kGatedBlock / 64) + uniform((int)threadIdx.x >> 6);
    if (wave >= L.blocks || *a.gate == 0) return;
    march_packets<1, true>(sdf_field(a.sdf, a.W, a.H), L, wave, a.emis4);
}

// The split march over a work list of (view, level) jobs, blocks in launch
// order as k_march_all's (the job list puts every view's top level first).
template <int SPEC, int M>
__global__ __launch_bounds__(kMarchBlock) void k_march_batch(const MarchJob *__restrict__ jobs,
                                                        const int *__restrict__ begins, int njobs)
{
    const int b = (int)blockIdx.x;
    const int j = batch_job(begins, njobs, b);
    const MarchJob J = jobs[j];
    march_all_body<SPEC, M>(J.sdf, J.W, J.H, J.L, b - begins[j], J.emis4);
}

// Persistent form of the split march.  March lengths differ by two orders of
// magnitude (most rays take 1-4 samples, rays grazing a surface up to a few
// hundred), so with one ray per lane a wave idles most lanes while its
// longest ray runs.  Here a grid of resident waves walks every ray of every
// level: the rays are cut into packets of 64 consecutive codes, numbered
// from the top level down (the longest rays first), and wave w owns packets
// w, w + n_waves, w + 2 n_waves, ... (an even mix of levels and image
// regions per wave).  Each lane holds its current ray and the next one,
// prepared ahead (its direction load issued an iteration or more before the
// ray starts, so starting it costs no dependent load): every iteration a lane
// whose ray ended takes its prepared one, the lanes without a prepared ray
// take the next entries of the wave's packet sequence (a ballot and a lane
// rank; the position in the sequence is a scalar, no memory atomics), and
// every busy lane takes one march round.  Each ray's samples, and so every
// code, are those of k_march_all; only the order of the rays differs.
template <int SPEC>
__global__ __launch_bounds__(kBlock) void k_march_persist(MarchAllArgs a)
{
    // per-level constants, indexed per lane (a lane's ray may be of any level)
    __shared__ int tab_i[RC_MAX_LEVELS][4];     // code_begin, PX, log2n, dir_off
    __shared__ float tab_f[RC_MAX_LEVELS][4];   // inv_px, spacing, t0, t1
    if ((int)threadIdx.x < a.nlev) {
        const MarchLevel &L = a.lev[threadIdx.x];
        tab_i[threadIdx.x][0] = (int)L.code_begin;
        tab_i[threadIdx.x][1] = L.PX;
        tab_i[threadIdx.x][2] = L.log2n;
        tab_i[threadIdx.x][3] = L.dir_off;
        tab_f[threadIdx.x][0] = L.inv_px;
        tab_f[threadIdx.x][1] = L.spacing;
        tab_f[threadIdx.x][2] = L.t0;
        tab_f[threadIdx.x][3] = L.t1;
    }
    __syncthreads();
    const SdfField f = sdf_field(a.sdf, a.W, a.H);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6));
    const uint32_t np = a.n_packets, nw = a.n_waves;
    // this wave's sequence length (waves past n_waves in the last workgroup have none)
    const uint32_t vend = (wave < nw && wave < np) ? ((np - 1 - wave) / nw + 1) * 64 : 0;
    uint32_t vnext = 0;  // wave-uniform
    Ray r = ray_begin(0.f, 0.f, 0.f, 0.f, 0.f, 0.f, false);
    float t1 = 0.f;
    uint32_t out = 0;
    bool have = false;
    // the prepared next ray
    float ncx = 0.f, ncy = 0.f, nt0 = 0.f, nt1 = 0.f;
    float2 ndir = make_float2(0.f, 0.f);
    uint32_t nout = 0;
    bool have_n = false;
    for (;;) {
        if (!have && have_n) {
            r = ray_begin(ncx, ncy, ndir.x, ndir.y, nt0, nt1, true);
            t1 = nt1;
            out = nout;
            have = true;
            have_n = false;
        }
        const uint64_t want = __ballot(!have_n);
        if (want != 0 && vnext < vend) {
            const uint32_t rank =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(want >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)want, 0u));
            const uint32_t v = vnext + rank;
            if (!have_n && v < vend) {
                const uint32_t pc = np - 1 - (wave + (v >> 6) * nw);  // packet in code order
                const uint32_t ray = pc * 64 + (v & 63);
                if (ray < a.total_rays) {
                    int lv = 0;  // levels are top first; code_begin falls with the level
#pragma unroll
                    for (int j = 0; j < RC_MAX_LEVELS; ++j)
                        if (j < a.nlev && ray < a.lev[j].code_begin) lv = j + 1;
                    const int rr = (int)(ray - (uint32_t)tab_i[lv][0]);
                    const int PX = tab_i[lv][1], log2n = tab_i[lv][2];
                    const int k = rr & ((1 << log2n) - 1), probe = rr >> log2n;
                    int py = (int)((float)probe * tab_f[lv][0]);
                    int px = probe - py * PX;
                    if (px < 0) { --py; px += PX; }
                    else if (px >= PX) { ++py; px -= PX; }
                    ndir = a.dirs_base[tab_i[lv][3] + k];  // used when the ray starts
                    const float sp = tab_f[lv][1];
                    ncx = ((float)px + 0.5f) * sp;
                    ncy = ((float)py + 0.5f) * sp;
                    nt0 = tab_f[lv][2];
                    nt1 = tab_f[lv][3];
                    nout = ray;
                    have_n = true;
                }
            }
            vnext += (uint32_t)__builtin_popcountll(want);
        }
        if (!__any(have || have_n)) {
            if (vnext >= vend) break;
            continue;
        }
        if (have) {
            ray_round<SPEC>(r, f, t1);
            if (!r.alive) {
                a.codes_base[out] = r.code;
                have = false;
            }
        }
    }
}

// For every slot of a level's split march, its ray's canonical index gets the
// slot number: the packets of the march's own waves, placed as it places them
// (parity readback).
__global__ __launch_bounds__(kMarchBlock) void k_ray_decode(MarchLevel l, int m, int64_t *__restrict__ index)
{
    const RayOrder o = ray_order(l, (int)threadIdx.x);
    const Packets p = wave_packets(l, (int)blockIdx.x, m);
    for (int T = p.first; T < p.end; T += p.step) {
        int px, py;
        uint32_t at;
        if (ray_place(o, l, T, px, py, at)) index[at + o.lat] = (int64_t)T * 64 + o.lane;
    }
}

template <Storage S>
__global__ __launch_bounds__(kBlock) void k_to_f32(const void *__restrict__ in, size_t texels, float4 *__restrict__ out)
{
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < texels) out[i] = Texel<S>::unpack(((const typename Texel<S>::T *)in)[i]);
}

int tile_kd(int shape)
{
    return shape == TILE_8x8x4 ? 4 : shape == TILE_4x4x16 ? 16 : shape == TILE_2x2x64 ? 64 : shape == TILE_8x4x8 ? 8 : 256;
}
int tile_tx(int shape)
{
    return shape == TILE_8x8x4 || shape == TILE_8x4x8 ? 8 : shape == TILE_4x4x16 ? 4 : shape == TILE_2x2x64 ? 2 : 1;
}
int tile_ty(int shape) { return shape == TILE_8x4x8 ? 4 : tile_tx(shape); }

template <int TX, int TY, int KD, int RPT, Storage S>
static void launch_level_shape(const LevelArgs &a, hipStream_t s)
{
    const int blocks = ((a.PX + TX - 1) / TX) * ((a.PY + TY * RPT - 1) / (TY * RPT)) * (a.N / KD);
    if (a.codes) {
        hipLaunchKernelGGL((k_level<TX, TY, KD, RPT, S, false, true>), dim3(blocks), dim3(kBlock), 0, s, a);
    } else {
        if (a.upper) hipLaunchKernelGGL((k_level<TX, TY, KD, RPT, S, true, false>), dim3(blocks), dim3(kBlock), 0, s, a);
        else hipLaunchKernelGGL((k_level<TX, TY, KD, RPT, S, false, false>), dim3(blocks), dim3(kBlock), 0, s, a);
    }
}

template <int RPT, Storage S>
static hipError_t launch_level_rpt(const LevelArgs &a, int shape, hipStream_t s)
{
    switch (shape) {
    case TILE_8x8x4: launch_level_shape<8, 8, 4, RPT, S>(a, s); break;
    case TILE_4x4x16: launch_level_shape<4, 4, 16, RPT, S>(a, s); break;
    case TILE_2x2x64: launch_level_shape<2, 2, 64, RPT, S>(a, s); break;
    case TILE_1x1x256: launch_level_shape<1, 1, 256, RPT, S>(a, s); break;
    case TILE_8x4x8: launch_level_shape<8, 4, 8, RPT, S>(a, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <Storage S>
static hipError_t launch_level_st(const LevelArgs &a, int shape, int rpt, hipStream_t s)
{
    if (tile_kd(shape) > a.N) return hipErrorInvalidValue;
    if (a.codes && a.upper) {
        const dim3 grid(merge_blocks(a.PX, a.PY, a.N));
        if (a.gate) {
            if (a.N < 64) hipLaunchKernelGGL((k_merge<S, true, true>), grid, dim3(kBlock), 0, s, a);
            else hipLaunchKernelGGL((k_merge<S, false, true>), grid, dim3(kBlock), 0, s, a);
        } else {
            if (a.N < 64) hipLaunchKernelGGL((k_merge<S, true, false>), grid, dim3(kBlock), 0, s, a);
            else hipLaunchKernelGGL((k_merge<S, false, false>), grid, dim3(kBlock), 0, s, a);
        }
        return hipGetLastError();
    }
    switch (rpt) {
    case 1: return launch_level_rpt<1, S>(a, shape, s);
    case 2: return launch_level_rpt<2, S>(a, shape, s);
    case 4: return launch_level_rpt<4, S>(a, shape, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_level(const LevelArgs &a, Storage st, int shape, int rpt, hipStream_t s)
{
    switch (st) {
    case Storage::F32: return launch_level_st<Storage::F32>(a, shape, rpt, s);
    case Storage::F16: return launch_level_st<Storage::F16>(a, shape, rpt, s);
    case Storage::BF16: return launch_level_st<Storage::BF16>(a, shape, rpt, s);
    }
    return hipErrorInvalidValue;
}

template <Storage S>
static hipError_t launch_level0_st(const LevelArgs &a, float *irr, float *dbg, hipStream_t s)
{
    const int blocks = level0_blocks(a.PX, a.PY);
    if (a.upper) hipLaunchKernelGGL((k_level0<S, true>), dim3(blocks), dim3(kBlock), 0, s, a, irr, dbg);
    else hipLaunchKernelGGL((k_level0<S, false>), dim3(blocks), dim3(kBlock), 0, s, a, irr, dbg);
    return hipGetLastError();
}

hipError_t launch_level0_gather(const LevelArgs &a, Storage st, float *irr, float *dbg, hipStream_t s)
{
    switch (st) {
    case Storage::F32: return launch_level0_st<Storage::F32>(a, irr, dbg, s);
    case Storage::F16: return launch_level0_st<Storage::F16>(a, irr, dbg, s);
    case Storage::BF16: return launch_level0_st<Storage::BF16>(a, irr, dbg, s);
    }
    return hipErrorInvalidValue;
}

template <int SPEC>
static hipError_t launch_march_all_spec(const MarchAllArgs &a, int m, int blocks, hipStream_t s)
{
    const dim3 grid(blocks, a.nlev);
    switch (m) {
    case 1: hipLaunchKernelGGL((k_march_all<SPEC, 1>), grid, dim3(kMarchBlock), 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_march_all<SPEC, 2>), grid, dim3(kMarchBlock), 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_march_all<SPEC, 4>), grid, dim3(kMarchBlock), 0, s, a); break;
    case 8: hipLaunchKernelGGL((k_march_all<SPEC, 8>), grid, dim3(kMarchBlock), 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_march_persist(const MarchAllArgs &a, int spec, hipStream_t s)
{
    if (a.nlev < 1 || a.total_rays == 0 || a.n_waves == 0) return hipSuccess;
    const dim3 grid((a.n_waves + 3) / 4);
    switch (spec) {
    case 1: hipLaunchKernelGGL(k_march_persist<1>, grid, dim3(kBlock), 0, s, a); break;
    case 2: hipLaunchKernelGGL(k_march_persist<2>, grid, dim3(kBlock), 0, s, a); break;
    case 4: hipLaunchKernelGGL(k_march_persist<4>, grid, dim3(kBlock), 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_march_all(const MarchAllArgs &a, int spec, int m, hipStream_t s)
{
    if (a.nlev < 1) return hipSuccess;  // one-level frame: no level >= 1 to march
    int blocks = 0;
    for (int i = 0; i < a.nlev; ++i) blocks = a.lev[i].blocks > blocks ? a.lev[i].blocks : blocks;
    if (blocks <= 0) return hipSuccess;
    if (a.gate) {
        constexpr int waves = kGatedBlock / 64;
        hipLaunchKernelGGL(k_march_gated, dim3((blocks + waves - 1) / waves, a.nlev), dim3(kGatedBlock), 0, s, a);
        return hipGetLastError();
    }
    switch (spec) {
    case 1: return launch_march_all_spec<1>(a, m, blocks, s);
    case 2: return launch_march_all_spec<2>(a, m, blocks, s);
    case 4: return launch_march_all_spec<4>(a, m, blocks, s);
    }
    return hipErrorInvalidValue;
}



int level_blocks(int PX, int PY, int N, int shape, int rpt)
{
    const int tx = tile_tx(shape), ty = tile_ty(shape) * rpt, kd = tile_kd(shape);
    return ((PX + tx - 1) / tx) * ((PY + ty - 1) / ty) * (N / kd);
}

int level0_blocks(int PX, int PY) { return ((PX + kL0TX - 1) / kL0TX) * ((PY + kL0TY - 1) / kL0TY); }

template <int SPEC>
static hipError_t launch_march_batch_spec(const BatchLaunch &b, int m, hipStream_t s)
{
    const MarchJob *j = (const MarchJob *)b.jobs;
    switch (m) {
    case 1: hipLaunchKernelGGL((k_march_batch<SPEC, 1>), dim3(b.blocks), dim3(kMarchBlock), 0, s, j, b.begins, b.njobs); break;
    case 2: hipLaunchKernelGGL((k_march_batch<SPEC, 2>), dim3(b.blocks), dim3(kMarchBlock), 0, s, j, b.begins, b.njobs); break;
    case 4: hipLaunchKernelGGL((k_march_batch<SPEC, 4>), dim3(b.blocks), dim3(kMarchBlock), 0, s, j, b.begins, b.njobs); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_march_batch(const BatchLaunch &b, int spec, int m, hipStream_t s)
{
    if (b.blocks <= 0) return hipSuccess;
    switch (spec) {
    case 1: return launch_march_batch_spec<1>(b, m, s);
    case 2: return launch_march_batch_spec<2>(b, m, s);
    }
    return hipErrorInvalidValue;
}

template <int TX, int TY, int KD, int RPT, Storage S>
static void launch_level_batch_shape(const BatchLaunch &b, bool from_codes, hipStream_t s)
{
    const LevelArgs *j = (const LevelArgs *)b.jobs;
    if (from_codes)
        hipLaunchKernelGGL((k_level_batch<TX, TY, KD, RPT, S, true>), dim3(b.blocks), dim3(kBlock), 0, s, j, b.begins,
                           b.njobs);
    else
        hipLaunchKernelGGL((k_level_batch<TX, TY, KD, RPT, S, false>), dim3(b.blocks), dim3(kBlock), 0, s, j, b.begins,
                           b.njobs);
}

template <int RPT, Storage S>
static hipError_t launch_level_batch_rpt(const BatchLaunch &b, int shape, bool from_codes, hipStream_t s)
{
    switch (shape) {
    case TILE_8x8x4: launch_level_batch_shape<8, 8, 4, RPT, S>(b, from_codes, s); break;
    case TILE_4x4x16: launch_level_batch_shape<4, 4, 16, RPT, S>(b, from_codes, s); break;
    case TILE_2x2x64: launch_level_batch_shape<2, 2, 64, RPT, S>(b, from_codes, s); break;
    case TILE_1x1x256: launch_level_batch_shape<1, 1, 256, RPT, S>(b, from_codes, s); break;
    case TILE_8x4x8: launch_level_batch_shape<8, 4, 8, RPT, S>(b, from_codes, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <Storage S>
static hipError_t launch_level_batch_st(const BatchLaunch &b, int shape, int rpt, bool from_codes, hipStream_t s)
{
    switch (rpt) {
    case 1: return launch_level_batch_rpt<1, S>(b, shape, from_codes, s);
    case 2: return launch_level_batch_rpt<2, S>(b, shape, from_codes, s);
    case 4: return launch_level_batch_rpt<4, S>(b, shape, from_codes, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_level_batch(const BatchLaunch &b, Storage st, int shape, int rpt, bool from_codes, hipStream_t s)
{
    if (b.blocks <= 0) return hipSuccess;
    switch (st) {
    case Storage::F32: return launch_level_batch_st<Storage::F32>(b, shape, rpt, from_codes, s);
    case Storage::F16: return launch_level_batch_st<Storage::F16>(b, shape, rpt, from_codes, s);
    case Storage::BF16: return launch_level_batch_st<Storage::BF16>(b, shape, rpt, from_codes, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_level0_batch(const BatchLaunch &b, Storage st, hipStream_t s)
{
    if (b.blocks <= 0) return hipSuccess;
    const Level0Job *j = (const Level0Job *)b.jobs;
    switch (st) {
    case Storage::F32: hipLaunchKernelGGL(k_level0_batch<Storage::F32>, dim3(b.blocks), dim3(kBlock), 0, s, j, b.begins, b.njobs); break;
    case Storage::F16: hipLaunchKernelGGL(k_level0_batch<Storage::F16>, dim3(b.blocks), dim3(kBlock), 0, s, j, b.begins, b.njobs); break;
    case Storage::BF16: hipLaunchKernelGGL(k_level0_batch<Storage::BF16>, dim3(b.blocks), dim3(kBlock), 0, s, j, b.begins, b.njobs); break;
    }
    return hipGetLastError();
}

hipError_t launch_level_to_f32(const void *level, Storage st, size_t texels, float *out, hipStream_t s)
{
    const unsigned blocks = (unsigned)((texels + kBlock - 1) / kBlock);
    if (blocks == 0) return hipSuccess;
    switch (st) {
    case Storage::F32: hipLaunchKernelGGL(k_to_f32<Storage::F32>, dim3(blocks), dim3(kBlock), 0, s, level, texels, (float4 *)out); break;
    case Storage::F16: hipLaunchKernelGGL(k_to_f32<Storage::F16>, dim3(blocks), dim3(kBlock), 0, s, level, texels, (float4 *)out); break;
    case Storage::BF16: hipLaunchKernelGGL(k_to_f32<Storage::BF16>, dim3(blocks), dim3(kBlock), 0, s, level, texels, (float4 *)out); break;
    }
    return hipGetLastError();
}

bool march_map_legal(int level, int map)
{
    static const int kd_log[kMarchMaps] = {0, 4, 2, 3, 5, 0};
    return level >= 1 && map >= 0 && map < kMarchMaps && (map == 0 || (1 << kd_log[map]) <= num_dirs(level));
}

void march_level_map(MarchLevel &l, int map)
{
    // (tx_log, ty_log, kd_log) of each wave tile; canonical order is one probe
    // x 64 directions where a level has them
    static const int tile[kMarchMaps][3] = {{0, 0, 6}, {1, 1, 4}, {2, 2, 2}, {2, 1, 3}, {1, 0, 5}, {3, 3, 0}};
    l.map = map;
    l.tx_log = tile[map][0];
    l.ty_log = tile[map][1];
    l.kd_log = map == 0 && l.log2n < 6 ? 0 : tile[map][2];
    l.ntx = (l.PX + (1 << l.tx_log) - 1) >> l.tx_log;
    const int nty = (l.PY + (1 << l.ty_log) - 1) >> l.ty_log;
    l.rcp_ntx = (uint32_t)std::min<uint64_t>(((1ull << 32) + l.ntx - 1) / l.ntx, 0xFFFFFFFFull);
    l.slots = map == 0 ? (uint32_t)((int64_t)l.PX * l.PY * l.N)
                       : (uint32_t)((int64_t)l.ntx * nty * (l.N >> l.kd_log) * 64);
}

void march_level_blocks(MarchLevel &l, int speculation, int rays_per_lane, int64_t launch_slots, int max_waves)
{
    l.packets = 1;
    l.stride = 1;
    l.group_log = 31;
    l.probe = false;
    if (rays_per_lane == 1) {
        // few enough packets a wave that several times the 8,192 waves the chip
        // holds are left: with 1, 2, 4 and 8 a frame of 256x256 (4,096 packets) took
        // 32.2, 34.1, 38.4 and 48.2 us, 1283x717 (72,000) 89.6, 86.5, 87.9 and 93.8,
        // one scene of 1920x1080 (163,200) 133.1, 126.4, 125.7 and 130.0 and another
        // 127.4 with 2 and 138.1 with 4, 6 scenes of 2200x1240 (216,000) 166.4, 160.1,
        // 160.3 and 161.8, of 2560x1440 (351,000) 243.7, 228.6, 224.1 and 227.9,
        // 3840x2160 (783,000) 553.9, 517.0, 506.8 and 503.2, 16 views of 9.2 megapixels
        // 900, 828, 792 and 772
        const int64_t n = launch_slots >> 6;
        // below this the chip is not full, loads are free and the longest ray is all:
        // 8 scenes of lit boxes of 256x256 (4,096 packets) 32.7 us guessing always, 33.3
        // probing; 700x300 (16,400) 49.9 and 49.8, with a thousandth of the pixels lit
        // 58.0 and 52.9
        l.probe = n >= 16 << 10;
        l.packets = n < 48 << 10 ? 1 : n < 192 << 10 ? 2 : n < 512 << 10 || l.map == 0 ? 4 : 8;
        const int mine = (int)(((int64_t)l.slots + 63) >> 6);
        l.stride = std::max(1, (mine + l.packets - 1) / l.packets);
        // A launch of 8 in canonical order marches 8 parts of the image at a
        // time, and a field of 8 MB does not stay in an L2 of 4 MB: there 4,096
        // waves keep to 16,384 consecutive packets.  3840x2160 with a ten
        // thousandth and a thousandth of the pixels lit 1,736 and 2,954 us with
        // 8, 1,585 and 2,731 so (1,492 and 2,586 with one, before the tail
        // guessed), 16 scenes of lit boxes 524 us on average either way; with
        // groups of 512 they took 534, with 1,024 to 8,192 and 8 packets 524 to
        // 529.  7680x4320 2,261 us with 8, 2,231 so.
        if (n >= 512 << 10 && l.map == 0 && l.stride > 4096) {
            l.stride = 4096;
            l.group_log = 12;
        }
        const int group = l.stride * l.packets;
        l.blocks = (mine + group - 1) / group * l.stride;
        if (l.blocks > max_waves) {
            l.blocks = l.stride = max_waves;
            l.packets = (mine + max_waves - 1) / max_waves;
            l.group_log = 31;
        }
        return;
    }
    const int64_t per = (int64_t)kMarchBlock * rays_per_lane;
    l.blocks = (int)(((int64_t)l.slots + per - 1) / per);
}

hipError_t launch_ray_decode(const MarchLevel &l, int rays_per_lane, int64_t *index, hipStream_t s)
{
    if (l.blocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ray_decode, dim3(l.blocks), dim3(kMarchBlock), 0, s, l, rays_per_lane, index);
    return hipGetLastError();
}

}  // namespace rc
