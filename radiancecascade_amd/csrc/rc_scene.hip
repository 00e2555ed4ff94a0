// rc_scene.hip -- seeded synthetic box scenes and their analytic G-buffer.
//
// This is the producer of the benchmark input, not part of the timed pass.
// The reference loads OBJ scenes (src/primitives.rs:122-175) and has no
// emissive material (src/primitives.rs:75-83), so the scene is the project's
// own: a unit-cube room (albedo 0.75) with axis-aligned boxes, camera at the
// room centre looking along +z with up +y in the reference's look_to_rh frame
// (src/camera.rs:43-52) and a 60 degree vertical field of view as the fovy of
// perspective_rh (src/camera.rs:77-79).  Depth is the linear view-space depth.
//
// The raster is FP64 with contraction off (the library is compiled with
// -ffp-contract=off): each pixel's result is a fixed sequence of correctly
// rounded IEEE operations, so it is reproducible bit for bit on any IEEE host.
#include "rc_internal.hpp"

namespace rc {

static uint64_t splitmix64_next(uint64_t &state)
{
    uint64_t z = (state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

static double unit_draw(uint64_t &state) { return (double)(splitmix64_next(state) >> 11) * 0x1.0p-53; }

// Per box: centre x,y,z ~ U[0,1); edges ~ 0.1 + 0.3 U; albedo ~ 0.2 + 0.7 U.
// A box overlapping the open clear zone (0.35,0.65)^3 around the camera is
// redrawn.  Then the first n_emissive boxes draw radiance 1 + 9 U per channel.
void scene_generate(uint64_t seed, int n_boxes, int n_emissive, rc_box *boxes)
{
    uint64_t st = seed;
    for (int b = 0; b < n_boxes; ++b) {
        bool blocked = true;
        while (blocked) {
            double c[3], e[3], a[3];
            for (double &v : c) v = unit_draw(st);
            for (double &v : e) v = 0.1 + 0.3 * unit_draw(st);
            for (double &v : a) v = 0.2 + 0.7 * unit_draw(st);
            blocked = true;
            for (int j = 0; j < 3; ++j) {
                boxes[b].lo[j] = c[j] - 0.5 * e[j];
                boxes[b].hi[j] = c[j] + 0.5 * e[j];
                boxes[b].albedo[j] = a[j];
                boxes[b].emit[j] = 0.0;
                blocked = blocked && boxes[b].lo[j] < 0.65 && 0.35 < boxes[b].hi[j];
            }
        }
    }
    for (int b = 0; b < n_emissive; ++b)
        for (double &v : boxes[b].emit) v = 1.0 + 9.0 * unit_draw(st);
}

// A workgroup rasterises 64x16 pixels, a lane one column's 4 rows of its wave.
// A pixel's ray direction is (dx(x), dy(y), 1), so a box's slab distances along
// x depend on the column alone and along y on the row alone: the workgroup
// computes them once per column and row (two divisions each) into LDS, 32
// boxes at a time, and a pixel only compares.  The z slab needs no division.
// Boxes behind the camera are dropped from the list first, and a wave skips a
// box whose x and z slabs miss all of its columns (or lie beyond what they
// already hit): the rest of the test can only narrow the interval.  Every
// distance is the quotient the per-pixel test would form, and the comparisons
// are made in its order, so the result is the same bit for bit.
//
// FP64 division bounds it: 4 per pixel and box (6 with z) took 199 us at
// 1920x1080 with 32 boxes, this form 28 us.
constexpr int kRasterRows = 16, kRasterChunk = 32;

struct RasterArgs {
    double box[kRasterArgBoxes * 12];
};
static_assert(sizeof(RasterArgs) + 40 <= 4096 && sizeof(RasterArgs) + 40 + 12 * sizeof(double) > 4096, "what a launch holds");

struct Slab {
    double n, f;  // nearer and farther plane
};
__device__ inline Slab slab(double lo, double hi, double d)
{
    const double t1 = (lo - 0.5) / d, t2 = (hi - 0.5) / d;
    return t1 > t2 ? Slab{t2, t1} : Slab{t1, t2};
}
// max / min by comparison: a NaN plane (0 / 0) changes nothing
__device__ inline void narrow(double &tn, double &tf, const Slab &s)
{
    if (s.n > tn) tn = s.n;
    if (s.f < tf) tf = s.f;
}

__device__ __forceinline__ void raster_body(const double *__restrict__ boxes, int n, int W, int H,
                                            float *__restrict__ depth, float *__restrict__ albedo,
                                            float *__restrict__ emissive)
{
    __shared__ Slab sx[kRasterChunk][64], sy[kRasterChunk][kRasterRows], sz[kRasterChunk];
    __shared__ int list[RC_MAX_BOXES], list_n;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const double th = 1.0 / sqrt(3.0);
    const double aspect = (double)W / (double)H;
    auto dir_x = [&](int x) {
        const double ndc_x = (2.0 * ((double)x + 0.5)) / (double)W - 1.0;
        return -((ndc_x * th) * aspect);
    };
    auto dir_y = [&](int y) {
        const double ndc_y = 1.0 - (2.0 * ((double)y + 0.5)) / (double)H;
        return ndc_y * th;
    };
    const int x0 = (int)blockIdx.x * 64, y0 = (int)blockIdx.y * kRasterRows;
    const int x = x0 + lane;

    // the boxes that reach in front of the camera, in order
    if (wave == 0) {
        int m = 0;
        for (int b0 = 0; b0 < n; b0 += 64) {
            const int b = b0 + lane;
            const bool keep = b < n && !(slab(boxes[12 * b + 2], boxes[12 * b + 5], 1.0).f <= 0.0);
            const unsigned long long mask = __ballot(keep);
            if (keep) list[m + __popcll(mask & ((1ull << lane) - 1))] = b;
            m += __popcll(mask);
        }
        if (lane == 0) list_n = m;
    }

    // the room: its nearest wall along the ray
    double best[4];
    int obj[4];
    {
        const double dx = dir_x(x);
        double tx = __builtin_huge_val();
        if (dx > 0.0) tx = (1.0 - 0.5) / dx;
        else if (dx < 0.0) tx = (0.0 - 0.5) / dx;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double dy = dir_y(y0 + 4 * wave + j);
            double t = tx, ty = __builtin_huge_val();
            if (dy > 0.0) ty = (1.0 - 0.5) / dy;
            else if (dy < 0.0) ty = (0.0 - 0.5) / dy;
            if (ty < t) t = ty;
            if (0.5 < t) t = 0.5;  // the far wall: (1 - 1/2) / 1
            best[j] = t;
            obj[j] = -1;
        }
    }
    __syncthreads();
    const int m = list_n;
    for (int c0 = 0; c0 < m; c0 += kRasterChunk) {
        const int nc = min(kRasterChunk, m - c0);
        if (c0 > 0) __syncthreads();
        for (int i = tid; i < nc * 64; i += kBlock) {
            const double *bx = boxes + 12 * list[c0 + (i >> 6)];
            sx[i >> 6][i & 63] = slab(bx[0], bx[3], dir_x(x0 + (i & 63)));
        }
        for (int i = tid; i < nc * kRasterRows; i += kBlock) {
            const double *bx = boxes + 12 * list[c0 + i / kRasterRows];
            sy[i / kRasterRows][i % kRasterRows] = slab(bx[1], bx[4], dir_y(y0 + i % kRasterRows));
        }
        if (tid < nc) {
            const double *bx = boxes + 12 * list[c0 + tid];
            sz[tid] = slab(bx[2], bx[5], 1.0);
        }
        __syncthreads();
        for (int k = 0; k < nc; ++k) {
            const Slab cx = sx[k][lane], cz = sz[k];
            double an = -__builtin_huge_val(), af = __builtin_huge_val();
            narrow(an, af, cx);
            double wn = an, wf = af;
            narrow(wn, wf, cz);
            const double far = fmax(fmax(best[0], best[1]), fmax(best[2], best[3]));
            if (!__any(wn <= wf && wf > 0.0 && wn < far)) continue;
            const int b = list[c0 + k];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                double tn = an, tf = af;
                narrow(tn, tf, sy[k][4 * wave + j]);
                narrow(tn, tf, cz);
                if (tn <= tf && tn > 0.0 && tn < best[j]) {
                    best[j] = tn;
                    obj[j] = b;
                }
            }
        }
    }
    if (x >= W) return;
    const size_t plane = (size_t)W * H;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int y = y0 + 4 * wave + j;
        if (y >= H) break;
        const size_t p = (size_t)y * W + x;
        depth[p] = (float)(best[j] * 1.0);
        for (int c = 0; c < 3; ++c) {
            if (albedo) albedo[c * plane + p] = obj[j] < 0 ? 0.75f : (float)boxes[12 * obj[j] + 6 + c];
            emissive[c * plane + p] = obj[j] < 0 ? 0.0f : (float)boxes[12 * obj[j] + 9 + c];
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_raster(const double *__restrict__ boxes, int n, int W, int H,
                                                   float *__restrict__ depth, float *__restrict__ albedo,
                                                   float *__restrict__ emissive)
{
    raster_body(boxes, n, W, H, depth, albedo, emissive);
}

// A box list short enough to travel with the launch (4 KB of kernel
// arguments): no device allocation and no copy before the kernel.
__global__ __launch_bounds__(kBlock) void k_raster_args(RasterArgs r, int n, int W, int H, float *__restrict__ depth,
                                                        float *__restrict__ albedo, float *__restrict__ emissive)
{
    __shared__ double sb[kRasterArgBoxes * 12];
    for (int i = threadIdx.x; i < n * 12; i += kBlock) sb[i] = r.box[i];
    __syncthreads();
    raster_body(sb, n, W, H, depth, albedo, emissive);
}

hipError_t launch_raster_args(const rc_box *boxes, int n, int W, int H, float *depth, float *albedo, float *emissive,
                              hipStream_t stream)
{
    static_assert(sizeof(rc_box) == 12 * sizeof(double), "a box is 12 doubles");
    RasterArgs r;
    for (int i = 0; i < n; ++i) __builtin_memcpy(r.box + 12 * i, boxes + i, sizeof(rc_box));
    dim3 grid((W + 63) / 64, (H + kRasterRows - 1) / kRasterRows);
    hipLaunchKernelGGL(k_raster_args, grid, dim3(kBlock), 0, stream, r, n, W, H, depth, albedo, emissive);
    return hipGetLastError();
}

hipError_t launch_raster(const double *boxes_dev, int n, int W, int H, float *depth, float *albedo, float *emissive,
                         hipStream_t stream)
{
    dim3 grid((W + 63) / 64, (H + kRasterRows - 1) / kRasterRows);
    hipLaunchKernelGGL(k_raster, grid, dim3(kBlock), 0, stream, boxes_dev, n, W, H, depth, albedo, emissive);
    return hipGetLastError();
}

}  // namespace rc
