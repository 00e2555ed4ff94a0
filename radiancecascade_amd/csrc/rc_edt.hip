// rc_edt.hip -- the exact distance field: occupancy bits, per-column vertical
// distances and per-row lower envelopes.
//
// The reference has no distance field (its only pass is the forward raster,
// src/renderer.rs:559-613).  The field the march reads is the one-byte code
// (rc_common.hpp) of d = sqrt(d^2), where
//   d^2(x, y) = min over occupied (x', y') of (x - x')^2 + (y - y')^2
// is the exact squared Euclidean distance transform of the occupancy (the
// occupancy rule of the seed kernel).  It is computed in its separable form
// (Felzenszwalb & Huttenlocher, "Distance Transforms of Sampled Functions",
// Theory of Computing 8, 2012, who build the row envelope with a stack):
//   g(x, y)   = min |y - y'| over occupied (x, y')          (per column)
//   d^2(x, y) = min over x' of (x - x')^2 + g(x', y)^2       (per row)
// d^2 is unique, so any exact method gives the same field; the kernels below
// are built for a 64-wide SIMT machine, not after that stack algorithm:
//   k_occ_bits : the occupancy of 64 x 64-pixel blocks as column words,
//                bits[y / 64][x] bit y % 64 (one ballot-free LDS transpose of
//                16 waves' 4-row nibbles), and the interleaved emission of
//                occupied pixels for the merge kernels;
//   k_edt_ends : per 64-row band and column, the nearest occupied rows above
//                and below the band (one sweep per column and direction, 8
//                words in flight): with the band's word they give g(x, y) in
//                a few bit operations, so g itself is never stored;
//   k_edt_rows : one workgroup per row, the row's g (from the words and the
//                band ends) in LDS.  The smallest argmin
//                opt(x) of (x - x')^2 + g(x')^2 never decreases with x (for
//                x1 < x2 and j < opt(x1), f_j(x2) - f_opt(x2) = f_j(x1) -
//                f_opt(x1) + 2 (x2 - x1)(opt - j) > 0), so it is found by divide
//                and conquer, each level between the argmins the earlier ones
//                fixed: over blocks of 8 candidates for rows up to 8192 pixels
//                (edt_row_blocks), pair by pair beyond (edt_row_body).
// Every step is exact integer arithmetic, so the field equals any exact
// transform's bit for bit.
#include <type_traits>

#include "rc_internal.hpp"

namespace rc {

constexpr uint32_t kGNone = 0xFFFFu;          // g of a column with no occupied pixel
constexpr int kOccBlock = 1024;               // k_occ_bits: 16 waves x 4 rows = 64 rows
constexpr int kRowLanes = 256;                // edt_row_body: lanes per row (4 waves)
// g of an empty column in the row kernel's LDS: its square (~2^30) is above
// every real value dx^2 + g^2 <= 2 * 16383^2 < 2^29 and dx^2 + 32767^2 < 2^32,
// so the pair value needs no clamp
constexpr uint32_t kGEmpty = 32767u;

__host__ __device__ inline int edt_bands(int H) { return (H + 63) >> 6; }
size_t edt_bits_bytes(int W, int H) { return (size_t)edt_bands(H) * W * sizeof(uint64_t); }
size_t edt_ends_bytes(int W, int H) { return 2 * (size_t)edt_bands(H) * W * sizeof(uint16_t); }

// ---- occupancy as column words --------------------------------------------
__device__ __forceinline__ void occ_bits_body(const float *__restrict__ depth, const DepthConv &dc,
                                              const float *__restrict__ emissive, uint64_t *__restrict__ bits,
                                              float4 *__restrict__ emis4, int W, int H, int bx_count, int b)
{
    __shared__ uint8_t nib[16][64];
    const int lane = (int)(threadIdx.x & 63), w = (int)(threadIdx.x >> 6);
    const int x = (b % bx_count) * 64 + lane;
    const int band = b / bx_count;
    const int y0 = band * 64 + 4 * w;
    uint32_t m = 0;
    if (x < W && y0 < H) {
        bool occ[4];
        float4 e[4];
        occupancy4(depth, dc, emissive, W, H, x, y0, occ, e);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (occ[j]) {
                m |= 1u << j;
                if (emis4) emis4[emis_index(x, y0 + j, W)] = e[j];
            }
    }
    nib[w][lane] = (uint8_t)m;
    __syncthreads();
    if (w == 0 && x < W) {
        uint64_t word = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) word |= (uint64_t)nib[k][lane] << (4 * k);
        bits[(size_t)band * W + x] = word;
    }
}

__global__ __launch_bounds__(kOccBlock) void k_occ_bits(const float *__restrict__ depth, DepthConv dc,
                                                        const float *__restrict__ emissive,
                                                        uint64_t *__restrict__ bits, float4 *__restrict__ emis4, int W,
                                                        int H, int bx_count, const int *gate)
{
    if (gate && *gate == 0) return;
    occ_bits_body(depth, dc, emissive, bits, emis4, W, H, bx_count, xcd_band(blockIdx.x, gridDim.x));
}

__global__ __launch_bounds__(kOccBlock) void k_occ_batch(const OccJob *__restrict__ jobs,
                                                         const int *__restrict__ begins, int njobs)
{
    const int b = xcd_band(blockIdx.x, gridDim.x);
    const int j = batch_job(begins, njobs, b);
    const OccJob &J = jobs[j];
    occ_bits_body(J.depth, J.dc, J.emissive, J.bits, J.emis4, J.W, J.H, J.bx_count, b - begins[j]);
}

// ---- band ends -------------------------------------------------------------
// For every 64-row band w and column x, the nearest occupied row above the
// band and below it: ends[w][x] (rows < 64 w) and ends[nb + w][x] (rows >=
// 64 (w + 1)), 0xFFFF for none.  One lane sweeps one column, down for the
// rows above (lanes [0, W)) or up for the rows below (lanes [W, 2W)), its
// band words loaded 8 at a time.  With the band's own word, these give any
// pixel's vertical distance g in a few bit operations (edt_g).
__device__ __forceinline__ void edt_ends_body(const uint64_t *__restrict__ bits, uint16_t *__restrict__ ends, int W,
                                              int H, int i)
{
    const int nb = edt_bands(H);
    if (i >= 2 * W) return;
    const bool down = i < W;
    const int x = down ? i : i - W;
    uint32_t near = kGNone;  // the occupied row nearest the band boundary reached so far
    for (int k0 = 0; k0 < nb; k0 += 8) {
        uint64_t v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int w = down ? k0 + k : nb - 1 - (k0 + k);
            v[k] = k0 + k < nb ? bits[(size_t)w * W + x] : 0ull;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (k0 + k >= nb) break;
            const int w = down ? k0 + k : nb - 1 - (k0 + k);
            ends[(size_t)(down ? w : nb + w) * W + x] = (uint16_t)near;
            if (v[k]) near = (uint32_t)(down ? w * 64 + 63 - __builtin_clzll(v[k]) : w * 64 + __builtin_ctzll(v[k]));
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_edt_ends(const uint64_t *__restrict__ bits, uint16_t *__restrict__ ends,
                                                     int W, int H, const int *gate)
{
    if (gate && *gate == 0) return;
    edt_ends_body(bits, ends, W, H, (int)(blockIdx.x * kBlock + threadIdx.x));
}

__global__ __launch_bounds__(kBlock) void k_ends_batch(const EndsJob *__restrict__ jobs,
                                                       const int *__restrict__ begins, int njobs)
{
    const int b = (int)blockIdx.x;
    const int j = batch_job(begins, njobs, b);
    const EndsJob &J = jobs[j];
    edt_ends_body(J.bits, J.ends, J.W, J.H, (b - begins[j]) * kBlock + (int)threadIdx.x);
}

// Vertical distance of pixel (x, y) to the nearest occupied pixel of its
// column (kGNone: the column has none) from the band's word, else the band
// ends (r = y % 64).
__device__ __forceinline__ uint32_t edt_g_of(uint64_t word, uint32_t ua, uint32_t db, int r, int y)
{
    const uint64_t le = word & ((2ull << r) - 1);  // rows <= r of the band (all 64 for r = 63)
    const uint64_t ge = word >> r;                 // rows >= r
    // both candidates, then a select (no branch for the loads to sink into;
    // the sentinel bits keep clz / ctz defined, their value unused then)
    const uint32_t up_in = (uint32_t)(r - 63 + __builtin_clzll(le | 1ull));
    const uint32_t dn_in = (uint32_t)__builtin_ctzll(ge | (1ull << 63));
    const uint32_t up_out = ua != kGNone ? (uint32_t)y - ua : kGNone;
    const uint32_t dn_out = db != kGNone ? db - (uint32_t)y : kGNone;
    const uint32_t up = le ? up_in : up_out, dn = ge ? dn_in : dn_out;
    return up < dn ? up : dn;
}

// ---- per-row lower envelope -------------------------------------------------------
// floor(sqrt(d2)) for d2 < 2^29: the hardware square root (within an ulp, so
// within 0.01 of the root here) truncated, then one integer correction step
// each way, which is all the truncation can be off by.
__device__ __forceinline__ uint32_t edt_isqrt(uint32_t d2)
{
    uint32_t r = (uint32_t)__builtin_amdgcn_sqrtf((float)d2);  // r < 2^15: 24-bit squares
    r -= __umul24(r, r) > d2 ? 1u : 0u;
    r += __umul24(r + 1, r + 1) <= d2 ? 1u : 0u;
    return r;
}

// The argmin of a solved pixel x: the low 16 bits of its 64-bit key
// (value << 16 | argmin), read through a 16-bit view of the key array.
__device__ __forceinline__ int edt_opt(const uint16_t *key16, int x) { return key16[4 * x]; }
// Candidate range [lo, hi] of query q (at x = (2q + 1) s - 1) at a level of
// step s: the argmins the earlier levels fixed at x -+ s (0 and W - 1 beyond
// the ends).
__device__ __forceinline__ int edt_lo(int q, int s, const uint16_t *key16)
{
    return q == 0 ? 0 : edt_opt(key16, 2 * q * s - 1);
}
__device__ __forceinline__ int edt_hi(int q, int s, int W, const uint16_t *key16)
{
    return (2 * q + 2) * s > W ? W - 1 : edt_opt(key16, (2 * q + 2) * s - 1);
}

// ---- rows up to 8192 pixels: blocks of 8 candidates ---------------------------
// The same divide and conquer with 2^B-way levels (B = 1, 2 or 3): a level of
// step s solves x = (q 2^B + r) s - 1, r = 1 .. 2^B - 1, between the argmins
// fixed at x = q 2^B s - 1 and (q + 1) 2^B s - 1 (group q).  Candidates are
// taken in aligned blocks of 8: a group's blocks run from lo / 8 to hi / 8, so
// the (group, block) pairs form the same kind of staircase, item t of it being
// block t - q of the last group q with lo(q) / 8 + q <= t, and a lane takes one
// item at a time.  (A block may hold candidates outside [lo, hi]; they cannot
// be a smaller argmin, so nothing is clamped.)
//
// An item is straight-line code on two 16-byte LDS reads.  With h_j = g_j^2 +
// j^2, the value (x - j)^2 + g_j^2 is x^2 + h_j - 2 x j.  hs[j] holds (h_j +
// bias) << 3 | i for candidate j = 8 block + i, so hs[j] - 16 x i orders a
// block's candidates by value and then by index in one 32-bit word: a
// multiply-add each and half a v_min3 per candidate and query.  The bias W^2 +
// 14 W keeps it, and h_j - 2 x j, non-negative; h_j + bias < 2^29 for every
// image with W <= 8192 (an empty column has W^2 + H^2 in the place of g^2,
// above any real value).  Items of a query meet at its pixel by a 64-bit LDS
// atomic minimum of (h_j - 2 x j + bias) << 3 over j.  Atomics of one wave on
// one address take their turns (about 7 cycles each: half of the kernel's
// time), so a wave within one group reduces over its lanes and sends one, and
// otherwise the lanes start at different queries of their group.
//
// Bound by instruction issue: 8 x 2^B candidate pairs take about 25 x 2^B + 80
// instructions, where the pair-by-pair walk took 12 a pair and 18 more
// whenever any lane of a wave entered its next query.  1920x1080: 36.0 us pair
// by pair, 30.4 with blocks and plain atomics, 20.0 with the lanes' queries
// rotated and levels of 2 bits (20.4 with 3), 18.8 with 4 columns per lane in
// the first and last pass; 3840x2160: 124 -> 52 us.
constexpr int kRowBlocksMax = 8192;


__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v)
{
    // row_shr 1, 2, 4, 8, then row broadcasts: lane 63 holds the minimum
#define RC_MIN_DPP(ctrl, rows)                                                                                     \
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, ctrl, rows, 0xF, false))
    RC_MIN_DPP(0x111, 0xF);
    RC_MIN_DPP(0x112, 0xF);
    RC_MIN_DPP(0x114, 0xF);
    RC_MIN_DPP(0x118, 0xF);
    RC_MIN_DPP(0x142, 0xA);
    RC_MIN_DPP(0x143, 0xC);
#undef RC_MIN_DPP
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Keys are stored with a gap after every 8: the positions a level's search
// reads lie a power of two apart.  key_bytes: byte offset of the key of x = n -
// 1 for n a multiple of 2^lg (one multiply-add).
__device__ __forceinline__ int key_at(int x) { return x + (x >> 3); }
__device__ __forceinline__ int key_bytes(int n, int lg) { return lg >= 3 ? __mul24(n, 9) - 16 : 8 * n - 8; }
__device__ __forceinline__ int block_opt(const unsigned long long *key, int bytes)
{
    return *reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(key) + bytes);
}

template <int RL, int B>
__device__ __forceinline__ void edt_block_level(const uint32_t *hs, unsigned long long *key, int W, int ls)
{
    constexpr int R = (1 << B) - 1;
    const int lane = (int)(threadIdx.x & 63), wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int s = 1 << ls, lg = ls + B, rot = lane % R;
    const int ng = ((W >> ls) + R) >> B;  // groups whose first query lies in the row
    const int hi = (ng << lg) > W ? W - 1 : block_opt(key, key_bytes(ng << lg, lg));
    // key_bytes(m << lg, lg) = m * step - first
    const int step = lg >= 3 ? 9 << lg : 8 << lg, first = lg >= 3 ? 16 : 8;
    const int T = (hi >> 3) + ng;
    for (int t0 = wave * 64; t0 < T; t0 += RL) {
        const int t = min(t0 + lane, T - 1);  // lanes past the end repeat the last item
        // the last group starting at or before t: a lower bound of uniform width
        int a = 0;
        for (int n = ng; n > 1;) {
            const int h = n >> 1, m = a + h;
            if ((block_opt(key, __mul24(m, step) - first) >> 3) + m <= t) a = m;
            n -= h;
        }
        const int blk = t - a;
        const uint4 *h4 = reinterpret_cast<const uint4 *>(hs) + 2 * blk;
        const uint4 u = h4[0], v = h4[1];
        const uint32_t h[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        const int x1 = (a << lg) + s - 1;
        const int a0 = __builtin_amdgcn_readfirstlane(a);
        const bool one_group = a0 == __builtin_amdgcn_readlane(a, 63);
        // the lanes of a group start at different queries, so its atomics go
        // to R addresses at a time
        int rr = one_group ? 0 : rot;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int x = x1 + (rr << ls);
            const int nx = -(x << 4);  // |nx| < 2^20: 24-bit products
            rr = rr == R - 1 ? 0 : rr + 1;
            uint32_t bv = h[0];
#pragma unroll
            for (int i = 1; i < 8; ++i) bv = min(bv, h[i] + (uint32_t)__mul24(i, nx));
            const uint32_t arg = (bv & 7u) | (uint32_t)(8 * blk);
            const uint32_t val = (bv & ~7u) + (uint32_t)__mul24(8 * blk, nx);
            bool mine = x < W;
            if (one_group) {
                // smallest value, then the lowest lane (smallest block) holding it
                const uint32_t w = wave_min_u32(val);
                mine = mine && lane == __builtin_ctzll(__ballot(val == w));
            }
            // B = 3 is the last level: x = 8 a + rr, the key after a gaps
            const int bytes = B == 3 ? 72 * a + ((x & 7) << 3) : key_bytes(x + 1, ls);
            if (mine)
                atomicMin(reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(key) + bytes),
                          ((unsigned long long)val << 32) | arg);
        }
    }
    __syncthreads();
}

// v_ffbh_u32 / v_ffbl_b32: leading / trailing zeros, 0xFFFFFFFF for 0.
__device__ __forceinline__ uint32_t ffbh(uint32_t v)
{
    uint32_t r;
    asm("v_ffbh_u32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ uint32_t ffbl(uint32_t v)
{
    uint32_t r;
    asm("v_ffbl_b32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
// Vertical distance to the nearest occupied pixel of the column as edt_g_of's,
// above 2^14 for none: the minimum of the distances within the band (huge
// where there is no bit) and to the band ends, which are never nearer than an
// occupied row of the band.  HIGH: r >= 32.
template <bool HIGH>
__device__ __forceinline__ uint32_t block_g(uint64_t word, uint32_t ua, uint32_t db, int r, int y)
{
    const uint32_t lo = (uint32_t)word, hi = (uint32_t)(word >> 32), out_up = (uint32_t)y - ua, out_dn = db - (uint32_t)y;
    if (HIGH) {
        const uint32_t q = (uint32_t)r - 32;
        const uint32_t up = ffbh(hi & ((2u << q) - 1)) - (31 - q);  // rows 32 .. r
        const uint32_t up2 = __builtin_elementwise_add_sat(ffbh(lo), q + 1);
        return min(min(min(up, up2), out_up), min(ffbl(hi >> q), out_dn));
    }
    const uint32_t up = ffbh(lo & ((2u << r) - 1)) - (31 - (uint32_t)r);
    const uint32_t dn2 = __builtin_elementwise_add_sat(ffbl(hi), 32 - (uint32_t)r);
    return min(min(min(up, out_up), dn2), min(ffbl(lo >> r), out_dn));
}

// floor(sqrt(d2)) for d2 < 2^29: the hardware square root of the rounded
// float is within 0.0035 of the root, so with 2^-7 added its integer part is
// the root or one above it.
__device__ __forceinline__ uint32_t block_isqrt(uint32_t d2)
{
    const uint32_t r = (uint32_t)(__builtin_amdgcn_sqrtf((float)d2) + 0.0078125f);
    return r - (__umul24(r, r) > d2 ? 1u : 0u);
}

template <int WMAX, int RL>
__device__ __forceinline__ void edt_row_blocks(const uint64_t *__restrict__ bits, const uint16_t *__restrict__ ends,
                                               uint8_t *__restrict__ sdf, int W, int H, int y)
{
    static_assert(WMAX == 8 * RL, "a lane has two runs of 4 columns");
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2), aligned(8)));
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4), aligned(2)));
    __shared__ __attribute__((aligned(16))) uint32_t hs[WMAX];
    // (h_j - 2 x j + bias) << 35 | j of the smallest argmin j; all ones until solved
    __shared__ unsigned long long key[WMAX + WMAX / 8];
    const int tid = (int)threadIdx.x;
    const int nb = edt_bands(H);
    const uint32_t empty = (uint32_t)(W * W) + (uint32_t)(H * H), bias = (uint32_t)(W * W + 14 * W);
    {
        // the row's g, 4 consecutive columns a lane and run; both runs' loads
        // are issued before either is used
        const int w = y >> 6, r = y & 63;
        const uint64_t *brow = bits + (size_t)w * W;
        const uint16_t *urow = ends + (size_t)w * W, *drow = ends + (size_t)(nb + w) * W;
        uint64_t wd[2][4];
        uint32_t ua[2][4], db[2][4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int x0 = 4 * (tid + k * RL);
            if (x0 + 4 <= W) {
                const u64x2 a = *reinterpret_cast<const u64x2 *>(brow + x0);
                const u64x2 b = *reinterpret_cast<const u64x2 *>(brow + x0 + 2);
                const u16x4 u = *reinterpret_cast<const u16x4 *>(urow + x0);
                const u16x4 d = *reinterpret_cast<const u16x4 *>(drow + x0);
                wd[k][0] = a[0], wd[k][1] = a[1], wd[k][2] = b[0], wd[k][3] = b[1];
#pragma unroll
                for (int i = 0; i < 4; ++i) ua[k][i] = u[i], db[k][i] = d[i];
            } else if (x0 < W) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int x = min(x0 + i, W - 1);
                    wd[k][i] = brow[x];
                    ua[k][i] = urow[x];
                    db[k][i] = drow[x];
                }
            }
        }
        auto store = [&](auto high) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int x0 = 4 * (tid + k * RL);
                if (x0 < W) {
                    uint32_t h[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t x = (uint32_t)(x0 + i);
                        const uint32_t g = block_g<decltype(high)::value>(wd[k][i], ua[k][i], db[k][i], r, y);
                        const uint32_t g2 = g > 16383u ? empty : (uint32_t)__umul24(g, g);
                        h[i] = ((g2 + (uint32_t)__umul24(x, x) + bias) << 3) | (x & 7u);
                        if (x >= (uint32_t)W) h[i] = 0xFFFFFFFFu;  // beyond the row: never a minimum
                        key[key_at(x0) + i] = ~0ull;
                    }
                    *reinterpret_cast<uint4 *>(hs + x0) = make_uint4(h[0], h[1], h[2], h[3]);
                }
            }
        };
        if (r >= 32) store(std::true_type{});
        else store(std::false_type{});
        // the rest of the last block
        if (tid < 4 && (((W + 3) & ~3) & 4)) hs[((W + 3) & ~3) + tid] = 0xFFFFFFFFu;
    }
    __syncthreads();
    // K bits with 2^K > W: the last level 3, those above 2 each (their groups
    // are few and large, so a query costs more than a search), an odd one first
    const int K = 32 - __builtin_clz((uint32_t)W);
    int ls = K;
    if ((K & 1) == 0 || K < 3) {
        ls -= 1;
        edt_block_level<RL, 1>(hs, key, W, ls);
    }
    while (ls > 3) {
        ls -= 2;
        edt_block_level<RL, 2>(hs, key, W, ls);
    }
    if (ls == 3) edt_block_level<RL, 3>(hs, key, W, 0);
    else if (ls == 1) edt_block_level<RL, 1>(hs, key, W, 0);
    // the codes of 4 consecutive columns in one store (a strip's row is 16
    // consecutive bytes), 0 in the last strip's columns past W and in row H
    const uint32_t skip = (uint32_t)sdf_skip(H), row = (uint32_t)y << 4;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int x0 = 4 * (tid + k * RL);
        if (x0 < sdf_width(W)) {
            uint32_t word = 0;
            if (x0 < W) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t x = (uint32_t)(x0 + i);
                    const uint32_t d2 =
                        ((uint32_t)(key[key_at(x0) + i] >> 32) >> 3) + (uint32_t)__umul24(x, x) - bias;
                    // sdf_code_of_distance: 128 + (d - 128) / 16 = (d + 1920) / 16, 255 from 2160 on
                    const uint32_t d = block_isqrt(d2), far = min((d + 1920u) >> 4, kSdfFar);
                    word |= (x0 + i >= W ? 0 : d2 >= empty ? kSdfFar : d < 128u ? d : far) << (8 * i);
                }
            }
            uint32_t *at = reinterpret_cast<uint32_t *>(sdf + (__umul24((uint32_t)x0 >> 4, skip) + (uint32_t)x0 + row));
            at[0] = word;
            if (y == H - 1) at[4] = 0;
        }
    }
}

// ---- wider rows ---------------------------------------------------------------
// Row y of a W-pixel image (W <= WMAX) by one workgroup of RL lanes.
// Consecutive queries of a level share an end (hi(q) = lo(q + 1)), so the
// level's (query, candidate) pairs form one staircase of T = hi(nq - 1) + nq
// steps: query q owns the steps [lo(q) + q, hi(q) + q], step t of it being
// candidate j = t - q.  The work per query is very uneven (a query whose
// neighbours' argmins lie on either side of a wide gap spans the gap), so
// the lanes take equal runs of steps instead: a lane finds the query of its
// first step by binary search on lo(q) + q (the argmins in LDS), walks its
// run in one loop of uniform trip count, keeping the first smallest value
// (ties go to the smallest candidate), and meets the other lanes of a query
// by a 64-bit LDS atomic minimum of (value << 16 | candidate) at the query's
// own pixel.  Every pixel is solved at exactly one level, so the keys start
// at all ones and need no reset between levels, and the next level reads the
// argmins straight from them: one barrier per level.
template <int WMAX, int RL>
__device__ __forceinline__ void edt_row_body(const uint64_t *__restrict__ bits, const uint16_t *__restrict__ ends,
                                             uint8_t *__restrict__ sdf, int W, int H, int y)
{
    __shared__ uint16_t gs[WMAX];
    __shared__ unsigned long long key[WMAX];  // key[x] = value << 16 | smallest argmin, all ones until solved
    const uint16_t *opt = reinterpret_cast<const uint16_t *>(key);
    const int tid = (int)threadIdx.x;
    const int nb = edt_bands(H);
    {
        // the row's g: every load of a batch of columns issued before any is
        // used (one round trip per batch, not one or two per column)
        constexpr int GB = 8;
        const int w = y >> 6, r = y & 63;
        const uint64_t *brow = bits + (size_t)w * W;
        const uint16_t *urow = ends + (size_t)w * W, *drow = ends + (size_t)(nb + w) * W;
        for (int x0 = tid; x0 < W; x0 += GB * RL) {
            uint64_t wd[GB];
            uint32_t ua[GB], db[GB];
#pragma unroll
            for (int i = 0; i < GB; ++i) {
                const int x = min(x0 + i * RL, W - 1);
                wd[i] = brow[x];
                ua[i] = urow[x];
                db[i] = drow[x];
            }
            // the values are pinned here, so the compiler neither sinks a
            // load into the branch below nor issues it again there
#pragma unroll
            for (int i = 0; i < GB; ++i) asm volatile("" : "+v"(wd[i]), "+v"(ua[i]), "+v"(db[i]));
#pragma unroll
            for (int i = 0; i < GB; ++i) {
                const int x = x0 + i * RL;
                if (x < W) {
                    gs[x] = (uint16_t)min(edt_g_of(wd[i], ua[i], db[i], r, y), kGEmpty);
                    key[x] = ~0ull;
                }
            }
        }
    }
    __syncthreads();
    const int K = 32 - __builtin_clz((uint32_t)W);  // smallest K with 2^K > W
    for (int k = 0; k < K; ++k) {
        const int ls = K - 1 - k, s = 1 << ls;
        const int nq = ((W >> ls) + 1) >> 1;  // odd multiples of s up to W
        const int T = edt_hi(nq - 1, s, W, opt) + nq;
        const int c = (T + RL - 1) / RL;
        const int t0 = tid * c, t1 = min(t0 + c, T);
        if (t0 < t1) {
            // the last query starting at or before t0: a lower bound of
            // uniform width (a + n <= nq throughout, so m <= nq - 1)
            int a = 0;
            for (int n = nq; n > 1;) {
                const int h = n >> 1, m = a + h;
                if (edt_opt(opt, (m << (ls + 1)) - 1) + m <= t0) a = m;  // lo(m) + m
                n -= h;
            }
            // branch-free values: |x - j| < 2^14 and g <= kGEmpty fit the
            // 24-bit multiplier, and dx^2 + g^2 the 32 bits
            int q = a, x = (2 * q + 1) * s - 1;
            int end = edt_hi(q, s, W, opt) + q + 1;  // the first step of query q + 1
            uint32_t bv = 0xFFFFFFFFu, bj = 0;
            // key = value << 16 | candidate from 32-bit halves (value < 2^30)
            auto flush = [&]() {
                atomicMin(&key[x], ((unsigned long long)(bv >> 16) << 32) | ((bv << 16) | bj));
            };
            // candidate j = t - q and dx = x - j carried step to step: the
            // next step of a query is j + 1, dx - 1; entering the next query
            // keeps j (t and q both advance) and moves x on by 2 s
            int j = t0 - q, dx = x - j;
            for (int t = t0; t < t1; ++t, ++j, --dx) {
                if (t >= end) {  // the run enters the next query (sizes >= 1: one step)
                    flush();
                    bv = 0xFFFFFFFFu;
                    ++q;
                    x += 2 * s;
                    --j;
                    dx += 2 * s + 1;
                    end = edt_hi(q, s, W, opt) + q + 1;
                }
                const uint32_t gj = gs[j], g2 = (uint32_t)__umul24(gj, gj);
                const uint32_t v = (uint32_t)__mul24(dx, dx) + g2;
                if (v < bv) {
                    bv = v;
                    bj = (uint32_t)j;
                }
            }
            flush();
        }
        __syncthreads();
    }
    for (int x = tid; x < W; x += RL) {
        const int j = edt_opt(opt, x);
        const uint32_t gj = gs[j];
        uint32_t code = kSdfFar;
        if (gj != kGEmpty) {  // |x - j| < 2^14 and g < 2^14: d^2 < 2^29
            const int dx = x - j;
            code = sdf_code_of_distance(edt_isqrt((uint32_t)__mul24(dx, dx) + (uint32_t)__umul24(gj, gj)));
        }
        sdf_store(sdf, x, y, W, H, code);
    }
}

// One row of an image that fits WMAX columns.
template <int WMAX, int RL>
__device__ __forceinline__ void edt_row(const uint64_t *__restrict__ bits, const uint16_t *__restrict__ ends,
                                        uint8_t *__restrict__ sdf, int W, int H, int y)
{
    if constexpr (WMAX <= kRowBlocksMax) edt_row_blocks<WMAX, RL>(bits, ends, sdf, W, H, y);
    else edt_row_body<WMAX, RL>(bits, ends, sdf, W, H, y);
}

// Lanes per row: one block of 8 candidates a lane (the upper levels' items are
// W / 8 and a few).  At 1920 columns 128 lanes took 38.6 and 512 lanes 21.2 us
// where 256 took 34.9 and 20.4 (without and with the queries rotated).
constexpr int rows_lanes(int wmax) { return wmax <= kRowBlocksMax ? wmax / 8 : kRowLanes; }

template <int WMAX>
__global__ __launch_bounds__(rows_lanes(WMAX)) void k_edt_rows(const uint64_t *__restrict__ bits,
                                                               const uint16_t *__restrict__ ends,
                                                               uint8_t *__restrict__ sdf, int W, int H,
                                                               const int *gate)
{
    if (gate && *gate == 0) return;
    edt_row<WMAX, rows_lanes(WMAX)>(bits, ends, sdf, W, H, xcd_band(blockIdx.x, gridDim.x));
}

template <int WMAX>
__global__ __launch_bounds__(rows_lanes(WMAX)) void k_rows_batch(const RowJob *__restrict__ jobs,
                                                                 const int *__restrict__ begins, int njobs)
{
    const int b = xcd_band(blockIdx.x, gridDim.x);
    const int j = batch_job(begins, njobs, b);
    const RowJob &J = jobs[j];
    edt_row<WMAX, rows_lanes(WMAX)>(J.bits, J.ends, J.sdf, J.W, J.H, b - begins[j]);
}

// ---- launchers ---------------------------------------------------------------------
int occ_blocks(int W, int H) { return ((W + 63) / 64) * edt_bands(H); }
int occ_bx(int W) { return (W + 63) / 64; }
int ends_blocks(int W) { return (2 * W + kBlock - 1) / kBlock; }
int edt_row_wmax(int W)
{
    int m = 512;
    while (m < W) m <<= 1;
    return m;
}

template <int WMAX>
static void launch_rows_t(const uint64_t *bits, const uint16_t *ends, uint8_t *sdf, int W, int H, hipStream_t s,
                          const int *gate)
{
    hipLaunchKernelGGL(k_edt_rows<WMAX>, dim3(H), dim3(rows_lanes(WMAX)), 0, s, bits, ends, sdf, W, H, gate);
}

hipError_t launch_edt(const float *depth, const DepthConv &dc, const float *emissive, uint64_t *bits, uint16_t *ends,
                      uint8_t *sdf, float4 *emis4, int W, int H, hipStream_t s, const int *gate, int stage)
{
    if (W < 1 || H < 1 || W > RC_MAX_DIM || H > RC_MAX_DIM) return hipErrorInvalidValue;
    const int bx = occ_bx(W);
    if (stage & 1)
        hipLaunchKernelGGL(k_occ_bits, dim3(occ_blocks(W, H)), dim3(kOccBlock), 0, s, depth, dc, emissive, bits, emis4,
                           W, H, bx, gate);
    if (stage & 2) {
        const uint64_t *cb = bits;
        hipLaunchKernelGGL(k_edt_ends, dim3(ends_blocks(W)), dim3(kBlock), 0, s, cb, ends, W, H, gate);
        switch (edt_row_wmax(W)) {
        case 512: launch_rows_t<512>(cb, ends, sdf, W, H, s, gate); break;
        case 1024: launch_rows_t<1024>(cb, ends, sdf, W, H, s, gate); break;
        case 2048: launch_rows_t<2048>(cb, ends, sdf, W, H, s, gate); break;
        case 4096: launch_rows_t<4096>(cb, ends, sdf, W, H, s, gate); break;
        case 8192: launch_rows_t<8192>(cb, ends, sdf, W, H, s, gate); break;
        default: launch_rows_t<16384>(cb, ends, sdf, W, H, s, gate); break;
        }
    }
    return hipGetLastError();
}

hipError_t launch_occ_batch(const BatchLaunch &b, hipStream_t s)
{
    if (b.blocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_occ_batch, dim3(b.blocks), dim3(kOccBlock), 0, s, (const OccJob *)b.jobs, b.begins, b.njobs);
    return hipGetLastError();
}

hipError_t launch_ends_batch(const BatchLaunch &b, hipStream_t s)
{
    if (b.blocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ends_batch, dim3(b.blocks), dim3(kBlock), 0, s, (const EndsJob *)b.jobs, b.begins, b.njobs);
    return hipGetLastError();
}

hipError_t launch_rows_batch(const BatchLaunch &b, int wmax, hipStream_t s)
{
    if (b.blocks <= 0) return hipSuccess;
    const RowJob *j = (const RowJob *)b.jobs;
    switch (wmax) {
    case 512:
        hipLaunchKernelGGL(k_rows_batch<512>, dim3(b.blocks), dim3(rows_lanes(512)), 0, s, j, b.begins, b.njobs);
        break;
    case 1024:
        hipLaunchKernelGGL(k_rows_batch<1024>, dim3(b.blocks), dim3(rows_lanes(1024)), 0, s, j, b.begins, b.njobs);
        break;
    case 2048:
        hipLaunchKernelGGL(k_rows_batch<2048>, dim3(b.blocks), dim3(rows_lanes(2048)), 0, s, j, b.begins, b.njobs);
        break;
    case 4096:
        hipLaunchKernelGGL(k_rows_batch<4096>, dim3(b.blocks), dim3(rows_lanes(4096)), 0, s, j, b.begins, b.njobs);
        break;
    case 8192:
        hipLaunchKernelGGL(k_rows_batch<8192>, dim3(b.blocks), dim3(rows_lanes(8192)), 0, s, j, b.begins, b.njobs);
        break;
    case 16384:
        hipLaunchKernelGGL(k_rows_batch<16384>, dim3(b.blocks), dim3(rows_lanes(16384)), 0, s, j, b.begins, b.njobs);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace rc
