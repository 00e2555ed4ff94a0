// rc_mlp.hip -- the surrogate MLP: BF16 MFMA forward (inference and
// training), backward, gradient reduction and Adam.
//
// Network (the project's own; the reference has no learned part):
// 64 -> 64 -> 64 -> 64 -> 64, ReLU on the hidden layers.  Outputs 0..47 are
// the level-1 far-field radiance (16 directions x rgb) in normalised units,
// output 48 the log of the predicted per-sample squared error (the per-tile
// fallback signal), outputs 49..63 padding.  Layer l computes
// z = bf16(a) . bf16(W) + b with FP32 accumulation on
// v_mfma_f32_32x32x16_bf16; the backward rounds each upstream gradient to
// bf16 before its two products (dW and dA) and keeps bias gradients in FP32.
//
// MFMA operand layout (32x32x16, wave64): lane l supplies row (l % 32) of A
// and column (l % 32) of B, each as 8 consecutive K elements starting at
// 8 * (l / 32); accumulator register v of lane l holds
// C[(v / 4) * 8 + (l / 32) * 4 + v % 4][l % 32].  Every operand is staged so
// that its 8 K elements are 16 contiguous bytes in LDS or global memory.
#include <string.h>

#include <vector>

#include "rc_internal.hpp"
#include "rc_shuffle.hpp"

namespace rc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// ---- parameter layout ---------------------------------------------------------
// FP32 master parameters: for l = 0..3, W_l [K_l][64] (input-major) then
// b_l [64].  bf16 copies: Wt_l [64][K_l] (output-major, forward B operand) and
// Wk_l [K_l][64] (input-major, backward B operand).
__host__ __device__ constexpr int mlp_k(int l) { return l == 0 ? kMlpIn : kMlpHid; }
__host__ __device__ constexpr int mlp_w_off(int l) { return l == 0 ? 0 : kMlpIn * 64 + (l - 1) * 64 * 64; }
__host__ __device__ constexpr int mlp_p_w(int l) { return mlp_w_off(l) + l * 64; }  // in the fp32 master vector
__host__ __device__ constexpr int mlp_p_b(int l) { return mlp_p_w(l) + mlp_k(l) * 64; }
static_assert(mlp_p_b(3) + 64 == kMlpParams, "parameter count");

__device__ inline uint16_t bf16_bits(float f) { return (uint16_t)f32_to_bf16_rne(f); }

// LDS row strides (elements) with 8 bf16 of padding: 16-byte aligned rows that
// do not all start on the same bank.
constexpr int kStrideHid = kMlpHid + 8;
constexpr int kStrideT = 32 + 8;         // transposed activations [feature][sample]

__device__ inline bf16x8 ld8(const uint16_t *p) { return *reinterpret_cast<const bf16x8 *>(p); }

// ---- inference over a feature matrix -------------------------------------------
// features [n][64] (already transformed, standardised here) -> z [n][64]
// fp32, 32 rows per wave with no exchange between waves.  Each layer is
// computed transposed, Z^T = W^T . A^T: a lane is one row of the batch (lane %
// 32), and the accumulators give it 8 groups of 4 consecutive outputs, the
// lane 32 further on the other 8.  Rounded to bf16 pairs, v_permlane32_swap
// between the two halves turns them into the next layer's operand, so
// activations never leave the registers.  The weight fragments are staged in
// LDS once per workgroup in the order the lanes read them.
//
// Bound by the feature and output rows (51 MB for 100,003 rows: 11 us at the
// rate of a large copy): 16 loads of 16 bytes a wave in flight, 4 waves per
// SIMD.  100,003 rows: 72.5 us with activations in LDS (2-byte stores, two
// barriers a layer), 13.4 us so.
constexpr int kInferLanes = 512;
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));  // any row address a caller may pass
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));

// Two floats rounded to bf16 (nearest even) in one v_cvt_pk_bf16_f32.
__device__ inline uint32_t bf16_pair(float lo, float hi)
{
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){lo, hi}, b2));
}

__global__ __launch_bounds__(kInferLanes, 4) void k_mlp_infer(MlpDev m, const float *__restrict__ feats, int n,
                                                              float *__restrict__ out)
{
    // fragment (layer, 32-output tile, 16-input chunk): 8 inputs of one output per lane
    __shared__ uintx4 wf[4][2][4][64];
    __shared__ __attribute__((aligned(16))) float bias_s[4 * 64], mean_s[kMlpIn], istd_s[kMlpIn];
    const int lane = threadIdx.x & 63, wave = (int)threadIdx.x >> 6, r = lane & 31, half = lane >> 5;
    for (int i = threadIdx.x; i < 4 * 2 * 4 * 64; i += kInferLanes) {
        const int ln = i & 63, k = (i >> 6) & 3, nt = (i >> 8) & 1, l = i >> 9;
        wf[l][nt][k][ln] = *reinterpret_cast<const uintx4 *>(m.wt + mlp_w_off(l) + (nt * 32 + (ln & 31)) * 64 + 16 * k +
                                                             8 * (ln >> 5));
    }
    if (threadIdx.x < 4 * 64) bias_s[threadIdx.x] = m.bias[threadIdx.x];
    if (threadIdx.x < kMlpIn) {
        mean_s[threadIdx.x] = m.in_mean[threadIdx.x];
        istd_s[threadIdx.x] = m.in_istd[threadIdx.x];
    }
    __syncthreads();
    const int blocks = (n + 31) / 32;
    for (int b = (int)blockIdx.x * (kInferLanes / 64) + wave; b < blocks; b += (int)gridDim.x * (kInferLanes / 64)) {
        const size_t row = (size_t)b * 32 + r;
        // a row past the end computes on the last row's features and stores nothing
        const float *f = feats + (row < (size_t)n ? row : (size_t)n - 1) * kMlpIn + 8 * half;
        floatx4 v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = *reinterpret_cast<const floatx4u *>(f + 16 * i);
            v[2 * i + 1] = *reinterpret_cast<const floatx4u *>(f + 16 * i + 4);
        }
        uintx4 x[4];  // the layer's input: 8 features of each 16-feature chunk
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int c = 16 * i + 8 * half + 4 * h;
                const floatx4 mu = *reinterpret_cast<const floatx4 *>(mean_s + c);
                const floatx4 sd = *reinterpret_cast<const floatx4 *>(istd_s + c);
                const floatx4 y = (v[2 * i + h] - mu) * sd;
                x[i][2 * h] = bf16_pair(y[0], y[1]);
                x[i][2 * h + 1] = bf16_pair(y[2], y[3]);
            }
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            asm volatile("" ::: "memory");  // the fragments are read per layer, not held over blocks (128 registers)
            floatx16 c[2] = {{}, {}};
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    c[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wf[l][nt][i][lane]),
                                                                    __builtin_bit_cast(bf16x8, x[i]), c[nt], 0, 0, 0);
            // outputs 32 nt + 8 q + 4 half + {0..3}
            uint32_t d[2][4][2];
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const floatx4 bb = *reinterpret_cast<const floatx4 *>(bias_s + l * 64 + nt * 32 + 8 * q + 4 * half);
                    floatx4 y = {c[nt][4 * q], c[nt][4 * q + 1], c[nt][4 * q + 2], c[nt][4 * q + 3]};
                    y = y + bb;
                    if (l == 3) {
                        if (row < (size_t)n)
                            *reinterpret_cast<floatx4u *>(out + row * kMlpOut + nt * 32 + 8 * q + 4 * half) = y;
                    } else {
                        d[nt][q][0] = bf16_pair(fmaxf(y[0], 0.0f), fmaxf(y[1], 0.0f));
                        d[nt][q][1] = bf16_pair(fmaxf(y[2], 0.0f), fmaxf(y[3], 0.0f));
                    }
                }
            if (l == 3) break;
            // chunk i of the next input: this half wants group 2 i + half whole,
            // of which it holds 4 outputs and the other half the other 4
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    const uintx2 sw = __builtin_amdgcn_permlane32_swap(d[i >> 1][2 * (i & 1)][w],
                                                                       d[i >> 1][2 * (i & 1) + 1][w], false, false);
                    x[i][w] = sw[0];
                    x[i][2 + w] = sw[1];
                }
        }
    }
}

// ---- training: forward + backward, per-workgroup gradient partials -----------
// A workgroup of 4 waves takes `nb` 32-sample blocks of the batch (sample ids
// from idx, or consecutive rows) and writes the FP32 sum of their gradients to
// partial[blockIdx.x][kMlpParams] and its loss sum.  Targets are normalised
// [n][48].  Waves 0 and 1 own the two 32-column tiles of every layer's
// output (and of the upstream gradient dA), their weight fragments held in
// registers; each of the 4 waves owns one 32x32 tile of every dW; wave 3 sums
// the bias gradients.
//
// What bounds it: 88 MFMAs a block take under a microsecond, the rest is the
// chain of about a dozen barrier-separated LDS steps, so the aim is many
// blocks in flight (64 KB of LDS: 2 workgroups, 8 waves per CU) and no global
// round trip inside a block; after that the 66.5 KB of partial sums each
// workgroup writes (34 MB for 16,384 samples).  The gradient is the sum of
// the 32-sample blocks' FP32 sums in block order, one partial each: the same bits
// whatever the grid.  Partials of several blocks would be fewer and another
// rounding of the same sum.  They are written in the accumulators' own order
// (part_to_master), 1 KB per store, and put in master order by the reduction.
// 16,384 samples: 85 us with one wave per block (weights read from L2 per
// product, scalar LDS copies), 20 us so.
constexpr int kTrainRow = 64 + 1, kTrainTgt = kMlpRad + 1;

// Where element i of a workgroup's partial belongs in the master vector: dW
// of layer l as 4 tiles of 32x32 in accumulator order ([tile][v / 4][lane][v %
// 4], tile 2 mt + nt: outputs 32 mt.., inputs 32 nt..), then the biases.
__device__ inline int part_to_master(int i)
{
    static_assert(kMlpIn == 64 && kMlpHid == 64, "square layers");
    if (i >= 4 * 4096) {
        const int b = i - 4 * 4096;
        return mlp_p_b(0) + (b >> 6) * (64 * 64 + 64) + (b & 63);
    }
    const int l = i >> 12, t = (i >> 10) & 3, q = (i >> 8) & 3, lane = (i >> 2) & 63, j = i & 3;
    const int o = (t >> 1) * 32 + 8 * q + 4 * (lane >> 5) + j, in = (t & 1) * 32 + (lane & 31);
    return mlp_p_w(0) + l * (64 * 64 + 64) + in * 64 + o;
}

__global__ __launch_bounds__(kBlock, 2) void k_mlp_train(MlpDev m, const float *__restrict__ feats,
                                                         const float *__restrict__ targets,
                                                         const int *__restrict__ idx, int batch, int nb,
                                                         float *__restrict__ partial, float *__restrict__ loss_part)
{
    __shared__ __attribute__((aligned(16))) uint16_t act[4][32 * kStrideHid];  // inputs of layers 0..3 [sample][feature]
    __shared__ __attribute__((aligned(16))) uint16_t actT[4][64 * kStrideT];   // the same [feature][sample]
    __shared__ __attribute__((aligned(16))) uint16_t g[32 * kStrideHid], gT[64 * kStrideT];
    __shared__ float zs[32 * kTrainRow];  // outputs, then the FP32 upstream gradient
    __shared__ float tg[32 * kTrainTgt];
    __shared__ float gerr[32];            // dL/dz_48
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int c32 = lane & 31, half = lane >> 5;
    const int oc = (wave & 1) * 32 + c32;  // the column of this lane in its wave's output tile
    bf16x8 wf[4][4], wb[3][4];
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (wave < 2) {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            bias[l] = m.bias[l * 64 + oc];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                wf[l][i] = ld8(m.wt + mlp_w_off(l) + oc * 64 + 16 * i + 8 * half);
                if (l > 0) wb[l - 1][i] = ld8(m.wk + mlp_w_off(l) + oc * 64 + 16 * i + 8 * half);
            }
        }
    }
    const float mean = m.in_mean[lane], istd = m.in_istd[lane];
    float *const part = partial + (size_t)blockIdx.x * kMlpParams;
    float loss_acc = 0.0f;
    const float inv_bn = 1.0f / ((float)batch * kMlpRad), inv_b = 1.0f / (float)batch;

    for (int bi = 0; bi < nb; ++bi) {
        const int s0 = ((int)blockIdx.x * nb + bi) * 32;
        // features (normalised) and targets of rows 8 wave .. 8 wave + 7, a
        // column per lane, all loads in flight at once.  Rows past the batch
        // are zero features with zero gradient.
        {
            float f[8], t[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int r = s0 + 8 * wave + j;
                const bool ok = r < batch;
                const size_t sid = ok ? (idx ? (size_t)idx[r] : (size_t)r) : 0;
                f[j] = ok ? feats[sid * kMlpIn + lane] : 0.0f;
                t[j] = ok && lane < kMlpRad ? targets[sid * kMlpRad + lane] : 0.0f;
            }
            uint32_t b[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                b[j] = s0 + 8 * wave + j < batch ? bf16_bits((f[j] - mean) * istd) : 0;
                act[0][(8 * wave + j) * kStrideHid + lane] = (uint16_t)b[j];
                if (lane < kMlpRad) tg[(8 * wave + j) * kTrainTgt + lane] = t[j];
            }
            *reinterpret_cast<uint4 *>(&actT[0][lane * kStrideT + 8 * wave]) =
                make_uint4(b[0] | b[1] << 16, b[2] | b[3] << 16, b[4] | b[5] << 16, b[6] | b[7] << 16);
        }
        __syncthreads();
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            if (wave < 2) {
                floatx16 c = {};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(act[l] + c32 * kStrideHid + 16 * i + 8 * half),
                                                                wf[l][i], c, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int row = 8 * q + 4 * half;
                    if (l == 3) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) zs[(row + j) * kTrainRow + oc] = c[4 * q + j] + bias[3];
                    } else {
                        uint32_t h[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            h[j] = bf16_bits(fmaxf(c[4 * q + j] + bias[l], 0.0f));
                            act[l + 1][(row + j) * kStrideHid + oc] = (uint16_t)h[j];
                        }
                        *reinterpret_cast<uint2 *>(&actT[l + 1][oc * kStrideT + row]) =
                            make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
                    }
                }
            }
            __syncthreads();
        }

        // loss and the error head's gradient: lanes 0..31 of wave 0 own one
        // sample each (FP32, fixed order)
        if (threadIdx.x < 32) {
            const bool ok = s0 + lane < batch;
            const float *z = zs + lane * kTrainRow, *t = tg + lane * kTrainTgt;
            float se = 0.0f;
#pragma unroll 16
            for (int c = 0; c < kMlpRad; ++c) {
                const float d = z[c] - t[c];
                se = fmaf(d, d, se);
            }
            const float de = z[kMlpErr] - logf(se * (1.0f / kMlpRad) + kMlpErrEps);
            if (ok) loss_acc += se * inv_bn + kMlpErrWeight * de * de * inv_b;
            gerr[lane] = ok ? kMlpErrWeight * 2.0f * de * inv_b : 0.0f;
        }
        __syncthreads();
        {
            // dL/dz4 of rows 8 wave.., a column per lane
            uint32_t b[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int r = 8 * wave + j;
                float gv = 0.0f;
                if (s0 + r < batch) {
                    if (lane < kMlpRad) gv = 2.0f * (zs[r * kTrainRow + lane] - tg[r * kTrainTgt + lane]) * inv_bn;
                    else if (lane == kMlpErr) gv = gerr[r];
                }
                zs[r * kTrainRow + lane] = gv;
                b[j] = bf16_bits(gv);
                g[r * kStrideHid + lane] = (uint16_t)b[j];
            }
            *reinterpret_cast<uint4 *>(&gT[lane * kStrideT + 8 * wave]) =
                make_uint4(b[0] | b[1] << 16, b[2] | b[3] << 16, b[4] | b[5] << 16, b[6] | b[7] << 16);
        }
        __syncthreads();

        // backward, layer 3 .. 0
#pragma unroll
        for (int l = 3; l >= 0; --l) {
            // dA_l = G (32 x 64) . W_l^T (64 x 64)
            floatx16 da = {};
            if (l > 0 && wave < 2) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    da = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(g + c32 * kStrideHid + 16 * i + 8 * half),
                                                                 wb[l > 0 ? l - 1 : 0][i], da, 0, 0, 0);
            }
            // dW^T tile [32 out][32 in] = G^T (32 samples) . A_l
            {
                const uint16_t *ga = gT + ((wave >> 1) * 32 + c32) * kStrideT + 8 * half;
                const uint16_t *ab = actT[l] + ((wave & 1) * 32 + c32) * kStrideT + 8 * half;
                floatx16 c = {};
#pragma unroll
                for (int k0 = 0; k0 < 32; k0 += 16)
                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(ga + k0), ld8(ab + k0), c, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    floatx4 *p = reinterpret_cast<floatx4 *>(part + l * 4096 + wave * 1024 + q * 256 + lane * 4);
                    const floatx4 v = {c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
                    *p = bi == 0 ? v : *p + v;
                }
            }
            // bias gradient: column sums in row order
            if (wave == 3) {
                float s = 0.0f;
#pragma unroll
                for (int r = 0; r < 32; ++r) s += zs[r * kTrainRow + lane];
                float *p = part + 4 * 4096 + l * 64 + lane;
                *p = bi == 0 ? s : *p + s;
            }
            __syncthreads();
            if (l == 0) break;
            if (wave < 2) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int row = 8 * q + 4 * half;
                    // the forward's ReLU output (stored, rounded) is > 0 exactly where the gradient passes
                    const uint2 hv = *reinterpret_cast<const uint2 *>(&actT[l][oc * kStrideT + row]);
                    const uint32_t h[4] = {hv.x & 0xFFFFu, hv.x >> 16, hv.y & 0xFFFFu, hv.y >> 16};
                    uint32_t b[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float gv = (h[j] != 0 && (h[j] & 0x8000u) == 0) ? da[4 * q + j] : 0.0f;
                        zs[(row + j) * kTrainRow + oc] = gv;
                        b[j] = bf16_bits(gv);
                        g[(row + j) * kStrideHid + oc] = (uint16_t)b[j];
                    }
                    *reinterpret_cast<uint2 *>(&gT[oc * kStrideT + row]) =
                        make_uint2(b[0] | b[1] << 16, b[2] | b[3] << 16);
                }
            }
            __syncthreads();
        }
    }
    // per-workgroup loss (lanes 0..31 of wave 0 hold row losses)
    if (wave == 0) {
        for (int o = 32; o >= 1; o >>= 1) loss_acc += __shfl_xor(loss_acc, o, 64);
        if (lane == 0) loss_part[blockIdx.x] = loss_acc;
    }
}

// One Adam step of master parameter i (Kingma & Ba 2015, bias-corrected), then
// its bf16 copies Wt (output-major) and Wk (input-major).
struct AdamStep {
    float lr, b1, b2, eps, c1, c2;
};
__device__ inline void adam_update(const MlpDev &m, int i, float gi, const AdamStep &a)
{
    const float mi = a.b1 * m.adam_m[i] + (1.0f - a.b1) * gi;
    const float vi = a.b2 * m.adam_v[i] + (1.0f - a.b2) * gi * gi;
    m.adam_m[i] = mi;
    m.adam_v[i] = vi;
    const float p = m.master[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
    m.master[i] = p;
    const int l = i / (64 * 64 + 64), e = i % (64 * 64 + 64);
    if (e < 64 * 64) {
        const uint16_t b = bf16_bits(p);
        m.wt[mlp_w_off(l) + (e & 63) * 64 + (e >> 6)] = b;
        m.wk[mlp_w_off(l) + e] = b;
    } else {
        m.bias[l * 64 + (e - 64 * 64)] = p;
    }
}

// Sum the workgroup partials in block order (deterministic), 64 elements per
// workgroup; the last workgroup sums the losses.  ADAM: the optimiser step of
// those elements follows in the same lanes (no gradient is stored).
//
// Bound by reading the partials (34 MB for 512 blocks): each workgroup's 512
// lanes keep 256 partials' 64 elements in flight (8 x 16 bytes a lane) and pass
// them through LDS to one wave, whose lanes add one element each in order
// while the next 256 partials are on their way.  One lane per element reading
// the partials itself had 65 workgroups with a few loads in flight: 512 blocks
// took 119 us, 10 us so (the Adam step included).
constexpr int kReduceLanes = 512, kReduceElems = 64, kReduceParts = 256;
static_assert(kMlpParams % kReduceElems == 0, "whole groups of elements");

template <bool ADAM>
__global__ __launch_bounds__(kReduceLanes) void k_mlp_reduce(const float *__restrict__ partial, int parts,
                                                             const float *__restrict__ loss_part,
                                                             float *__restrict__ grad, float *__restrict__ loss,
                                                             MlpDev m, AdamStep step)
{
    __shared__ __attribute__((aligned(16))) float sb[kReduceParts * kReduceElems];
    const int tid = (int)threadIdx.x;
    if (blockIdx.x == gridDim.x - 1) {
        // kBlock lanes, each a strided sum, then a fixed tree
        if (tid < kBlock) {
            float a = 0.0f;
            for (int i = tid; i < parts; i += kBlock) a += loss_part[i];
            sb[tid] = a;
        }
        __syncthreads();
        for (int w = kBlock / 2; w >= 1; w >>= 1) {
            if (tid < w) sb[tid] += sb[tid + w];
            __syncthreads();
        }
        if (tid == 0) *loss = sb[0];
        return;
    }
    const int e0 = (int)blockIdx.x * kReduceElems;
    const int p0 = tid >> 4, e4 = (tid & 15) * 4;
    constexpr int PER = kReduceParts / (kReduceLanes / 16);
    floatx4 v[PER];
    auto load = [&](int base) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int p = min(base + p0 + k * (kReduceLanes / 16), parts - 1);
            v[k] = *reinterpret_cast<const floatx4 *>(partial + (size_t)p * kMlpParams + e0 + e4);
        }
    };
    load(0);
    float s = 0.0f;
    for (int base = 0; base < parts; base += kReduceParts) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; ++k)
            *reinterpret_cast<floatx4 *>(sb + (p0 + k * (kReduceLanes / 16)) * kReduceElems + e4) = v[k];
        __syncthreads();
        if (base + kReduceParts < parts) load(base + kReduceParts);
        if (tid < kReduceElems) {
            const int n = min(kReduceParts, parts - base);
#pragma unroll 16
            for (int p = 0; p < n; ++p) s += sb[p * kReduceElems + tid];
        }
    }
    if (tid < kReduceElems) {
        const int i = part_to_master(e0 + tid);
        if (ADAM) adam_update(m, i, s, step);
        else grad[i] = s;
    }
}

// An Adam step of every parameter with a caller's gradient.
__global__ __launch_bounds__(kBlock) void k_mlp_adam(MlpDev m, const float *__restrict__ grad, AdamStep step)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < kMlpParams) adam_update(m, i, grad[i], step);
}

// Refresh the bf16 copies and biases from the master vector (after a load).
__global__ __launch_bounds__(kBlock) void k_mlp_refresh(MlpDev m)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= kMlpParams) return;
    const float p = m.master[i];
    for (int l = 0; l < 4; ++l) {
        const int K = mlp_k(l), w0 = mlp_p_w(l), b0 = mlp_p_b(l);
        if (i >= w0 && i < b0) {
            const int in = (i - w0) / 64, o = (i - w0) % 64;
            m.wt[mlp_w_off(l) + o * K + in] = bf16_bits(p);
            m.wk[mlp_w_off(l) + in * 64 + o] = bf16_bits(p);
        } else if (i >= b0 && i < b0 + 64) {
            m.bias[l * 64 + (i - b0)] = p;
        }
    }
}

// ---- the row order of an epoch ---------------------------------------------------
// The shuffle of rc_shuffle.hpp, a lane an element in each of its four steps.
// The sequential loop on the host is a chain of cache misses: about 1.3 ms for
// 524,288 rows (and 0.3 s for 16 M) with the upload; these four kernels take
// 64 us.
__global__ __launch_bounds__(kBlock) void k_shuffle_clear(int *__restrict__ head, int n)
{
    const int p = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (p < n) head[p] = -1;
}

// order[i] = j_i, step i linked into list j_i.
__global__ __launch_bounds__(kBlock) void k_shuffle_draw(uint64_t state, int n, int *__restrict__ order,
                                                         int *__restrict__ head, int *__restrict__ next)
{
    const int i = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (i >= n) return;
    if (i == 0) {
        order[0] = 0;
        return;
    }
    const int j = shuffle_target(state, n, i);
    order[i] = j;
    next[i] = atomicExch(&head[j], i);
}

// Each list in ascending order; a lane owns its list.
__global__ __launch_bounds__(kBlock) void k_shuffle_sort(int n, int *__restrict__ head, int *__restrict__ next)
{
    __shared__ int buf[kShuffleList][kBlock];
    const int p = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (p < n) shuffle_sort_list<kShuffleList>(p, head, next, &buf[0][threadIdx.x], kBlock);
}

__global__ __launch_bounds__(kBlock) void k_shuffle_resolve(int n, int *__restrict__ order,
                                                            const int *__restrict__ head, const int *__restrict__ next)
{
    const int i = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (i < n) shuffle_resolve(i, order, head, next);
}

hipError_t launch_shuffle(uint64_t state, size_t n, int *order, int *head, int *next, hipStream_t s)
{
    const dim3 g((unsigned)((n + kBlock - 1) / kBlock)), b(kBlock);
    hipLaunchKernelGGL(k_shuffle_clear, g, b, 0, s, head, (int)n);
    hipLaunchKernelGGL(k_shuffle_draw, g, b, 0, s, state, (int)n, order, head, next);
    hipLaunchKernelGGL(k_shuffle_sort, g, b, 0, s, (int)n, head, next);
    hipLaunchKernelGGL(k_shuffle_resolve, g, b, 0, s, (int)n, order, head, next);
    return hipGetLastError();
}

hipError_t launch_mlp_infer(const MlpDev &m, const float *feats, int n, float *out, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    // one 32-row block a wave up to 2 workgroups of 8 waves on each of 256 CUs, then several
    const int blocks = (n + 31) / 32, per = kInferLanes / 64;
    const int grid = (blocks + per - 1) / per;
    hipLaunchKernelGGL(k_mlp_infer, dim3(grid < 512 ? grid : 512), dim3(kInferLanes), 0, s, m, feats, n, out);
    return hipGetLastError();
}

hipError_t launch_mlp_train(const MlpDev &m, const float *feats, const float *targets, const int *idx, int batch,
                            int nb, float *partial, float *loss_part, int parts, hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_train, dim3(parts), dim3(kBlock), 0, s, m, feats, targets, idx, batch, nb, partial,
                       loss_part);
    return hipGetLastError();
}

hipError_t launch_mlp_reduce(const float *partial, const float *loss_part, int parts, float *grad, float *loss,
                             hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_reduce<false>, dim3(kMlpParams / kReduceElems + 1), dim3(kReduceLanes), 0, s, partial,
                       parts, loss_part, grad, loss, MlpDev{}, AdamStep{});
    return hipGetLastError();
}

hipError_t launch_mlp_reduce_adam(const MlpDev &m, const float *partial, const float *loss_part, int parts, float *loss,
                                  float lr, float b1, float b2, float eps, float c1, float c2, hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_reduce<true>, dim3(kMlpParams / kReduceElems + 1), dim3(kReduceLanes), 0, s, partial,
                       parts, loss_part, (float *)nullptr, loss, m, AdamStep{lr, b1, b2, eps, c1, c2});
    return hipGetLastError();
}

hipError_t launch_mlp_adam(const MlpDev &m, const float *grad, float lr, float b1, float b2, float eps, float c1,
                           float c2, hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_adam, dim3((kMlpParams + kBlock - 1) / kBlock), dim3(kBlock), 0, s, m, grad,
                       AdamStep{lr, b1, b2, eps, c1, c2});
    return hipGetLastError();
}

hipError_t launch_mlp_refresh(const MlpDev &m, hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_refresh, dim3((kMlpParams + kBlock - 1) / kBlock), dim3(kBlock), 0, s, m);
    return hipGetLastError();
}

}  // namespace rc
