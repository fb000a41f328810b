// kernels_reproj.hip -- the ProjAlign re-projector (AreTomo/ProjAlign/GReproj.cu,
// CCalcReproj.cpp) for gfx950: a projection at angle a is predicted from the
// nearby lower-tilt projections by a cos-weighted nearest-sample
// back-projection onto a 2x-wide slice followed by a forward projection at a.
//
// The reference runs one host loop iteration per image row (two launches
// and two copies per row) over a slice in memory.  Here no slice is formed:
// a ray reads each of its voxels once, so the voxel is evaluated where the ray
// needs it.  Coordinates are evaluated in FP64 with contraction off, from host
// FP64 tables, so every nearest-sample pick and every in/out decision is the
// one of the FP64 restatement; sums are FP64.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "atr_internal.h"

namespace atr {

// One workgroup: 64 output columns (lane = x) of RP_ROWS image rows; its four
// waves take a quarter of the ray's samples each.  Where a voxel samples the
// projections does not depend on the image row, so one evaluation of a
// sample's coordinates (about 10 FP64 operations per tilt and a division)
// serves all the rows, and the weight cos t cos(a - t) / sum cos(a - t) of a
// projection value is formed once for them: what is left per row, tilt and
// sample is a conversion and an FP64 FMA.  The columns that a segment of `seg`
// samples can reach are staged in LDS, four rows to a 16-byte entry.  A
// segment whose staged columns hold an empty value takes the general path,
// which counts each row's samples by itself.
//
// 1024^2 x 256, 8 reference tilts at 48 degrees: 0.68 ms (0.81 with the rays'
// sums written in the kernel's own body: 84 more reads of spilled scalars; 5.3
// with the slice formed in memory and read back, where every voxel of it cost
// its coordinates and a division).  Bound by VALU issue, busy 0.82 of the time:
// 59 instructions per sample and tilt, 16 of them FP64 arithmetic (8 for the
// rows, the others for coordinates), 8 conversions, the rest compares, picks,
// addresses and spilled scalars.
constexpr int RP_ROWS = 8;
constexpr int RP_WAVES = 4;
constexpr int RP_LDS = 52 * 1024;      // three workgroups per CU
constexpr int RP_LDS_MAX = 150 * 1024;

// The four waves' sums and counts of a ray, added in the ray's order, to its
// output pixel.
__device__ __forceinline__ void reproj_store(const ReprojArgs& a, const double (&sum)[RP_ROWS],
                                             const int (&cnt)[RP_ROWS], double* s_sum, int y0, int x,
                                             float* __restrict__ out)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int* s_cnt = (int*)(s_sum + RP_WAVES * RP_ROWS * 64);
#pragma unroll
    for (int r = 0; r < RP_ROWS; r++) {
        s_sum[(wave * RP_ROWS + r) * 64 + lane] = sum[r];
        s_cnt[(wave * RP_ROWS + r) * 64 + lane] = cnt[r];
    }
    __syncthreads();
    const int n_rows = min(RP_ROWS, a.proj_y - y0);
    for (int r = wave; r < n_rows; r += RP_WAVES) {
        double t = 0.0;
        int n = 0;
        for (int w = 0; w < RP_WAVES; w++) {
            t += s_sum[(w * RP_ROWS + r) * 64 + lane];
            n += s_cnt[(w * RP_ROWS + r) * 64 + lane];
        }
        if (x < a.proj_x)
            out[(size_t)(y0 + r) * a.proj_x + x] = ((float)n < a.min_count) ? kSentinel : (float)(t / n);
    }
}
constexpr int RP_SUMS = RP_WAVES * RP_ROWS * 64 * (int)(sizeof(double) + sizeof(int));

// N: number of reference tilts (their geometry stays in scalar registers).
template <int N>
__global__ __launch_bounds__(64 * RP_WAVES) void k_reproj(const float* __restrict__ projs,
                                                          ReprojArgs a, float* __restrict__ out)
{
#pragma clang fp contract(off)
    extern __shared__ float4 win[];    // [tilt][2][width]: rows 0-3, rows 4-7
    __shared__ int any_empty;
    __shared__ int s_low[N];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int xb = blockIdx.x * 64, x = xb + lane;
    const int y0 = blockIdx.y * RP_ROWS;
    const double fc = a.ray_cos, fs = a.ray_sin;
    const double hx = a.vol_x * 0.5, hz = a.vol_z * 0.5, cx = a.proj_x * 0.5;
    const int last = a.proj_x - 1;
    const double xp = x + 0.5 - a.proj_x * 0.5;
    const double tx = a.vol_x * 0.5 + a.ray * 0.5 * fs + xp / fc;
    const double tz = a.vol_z * 0.5 - a.ray * 0.5 * fc;
    // the rays at the two ends of the workgroup's columns
    const double txa = a.vol_x * 0.5 + a.ray * 0.5 * fs + (xb + 0.5 - a.proj_x * 0.5) / fc;
    const double txb = txa + 63.0 / fc;
    double sum[RP_ROWS];
    int cnt[RP_ROWS], plain_cnt = 0;
#pragma unroll
    for (int r = 0; r < RP_ROWS; r++) {
        sum[r] = 0.0;
        cnt[r] = 0;
    }
    for (int i0 = 0; i0 < a.ray; i0 += a.seg) {
        const int i1 = min(i0 + a.seg, a.ray);
        // first staged column of tilt k: two below the smallest coordinate of
        // the four corners of the segment's samples (a voxel's centre is at
        // most 0.71 from the sample)
        auto low = [&](int k) {
            const double c = a.cos_t[k], s = a.sin_t[k];
            const double ua = (txa - hx) * c, ub = (txb - hx) * c;
            const double d = fc * s - fs * c, b = (tz - hz) * s + cx;
            const double u = min(ua, ub) + b + min(i0 * d, (i1 - 1) * d);
            return min(max((int)floor(u) - 2, 0), last);
        };
        if (threadIdx.x == 0) any_empty = 0;
        if (threadIdx.x < N) s_low[threadIdx.x] = low(threadIdx.x);
        __syncthreads();
        int first_col[N];
#pragma unroll
        for (int k = 0; k < N; k++) first_col[k] = __builtin_amdgcn_readfirstlane(s_low[k]);
        bool empty = false;
#pragma unroll
        for (int k = 0; k < N; k++) {
            const int lo = first_col[k];
            const float* img = projs + (size_t)(a.first + k) * a.proj_y * a.proj_x;
            for (int i = threadIdx.x; i < 2 * a.width; i += 64 * RP_WAVES) {
                const int h = i >= a.width, col = i - h * a.width;
                const int g = min(lo + col, last);
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    v[r] = img[(size_t)min(y0 + 4 * h + r, a.proj_y - 1) * a.proj_x + g];
                    empty |= v[r] < kEmpty;
                }
                win[(k * 2 + h) * a.width + col] = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
        if (empty) any_empty = 1;
        __syncthreads();
        const bool plain = any_empty == 0;
        const int per = (i1 - i0 + RP_WAVES - 1) / RP_WAVES;
        const int ia = i0 + wave * per, ib = min(ia + per, i1);
        for (int i = ia; i < ib; i++) {
            const double px = tx - i * fs;
            const double pz = tz + i * fc;
            if (px < 0 || px >= a.vol_x || pz < 0 || pz >= a.vol_z) continue;
            const double fx = (int)px + 0.5 - a.vol_x * 0.5;
            const double fz = (int)pz + 0.5 - a.vol_z * 0.5;
            if (plain) {
                // the voxel is sum_k v_k c_k w_k / sum_k w_k over the tilts
                // that see it (nearly always all of them)
                double num[RP_ROWS], den = 0.0;
#pragma unroll
                for (int r = 0; r < RP_ROWS; r++) num[r] = 0.0;
#pragma unroll
                for (int k = 0; k < N; k++) {
                    const double u = fx * a.cos_t[k] + fz * a.sin_t[k] + cx;
                    if (u < 0 || u > last) continue;
                    const int col = min(max((int)u - first_col[k], 0), a.width - 1);
                    const float4 va = win[(k * 2) * a.width + col];
                    const float4 vb = win[(k * 2 + 1) * a.width + col];
                    const double w = a.cos_w[k];
                    den += a.weight[k];
                    num[0] = fma((double)va.x, w, num[0]);
                    num[1] = fma((double)va.y, w, num[1]);
                    num[2] = fma((double)va.z, w, num[2]);
                    num[3] = fma((double)va.w, w, num[3]);
                    num[4] = fma((double)vb.x, w, num[4]);
                    num[5] = fma((double)vb.y, w, num[5]);
                    num[6] = fma((double)vb.z, w, num[6]);
                    num[7] = fma((double)vb.w, w, num[7]);
                }
                if (den < 0.001) continue;
                double inv = a.inv_total;
                if (den != a.total) inv = 1.0 / den;
#pragma unroll
                for (int r = 0; r < RP_ROWS; r++) sum[r] = fma(num[r], inv, sum[r]);
                plain_cnt += 1;
            } else {
                double num[RP_ROWS], den[RP_ROWS];
#pragma unroll
                for (int r = 0; r < RP_ROWS; r++) num[r] = den[r] = 0.0;
#pragma unroll
                for (int k = 0; k < N; k++) {
                    const double u = fx * a.cos_t[k] + fz * a.sin_t[k] + cx;
                    if (u < 0 || u > last) continue;
                    const int col = min(max((int)u - first_col[k], 0), a.width - 1);
                    const float4 va = win[(k * 2) * a.width + col];
                    const float4 vb = win[(k * 2 + 1) * a.width + col];
                    const float v[RP_ROWS] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
#pragma unroll
                    for (int r = 0; r < RP_ROWS; r++) {
                        if (v[r] < kEmpty) continue;
                        num[r] += v[r] * a.cos_t[k] * a.weight[k];
                        den[r] += a.weight[k];
                    }
                }
#pragma unroll
                for (int r = 0; r < RP_ROWS; r++) {
                    if (den[r] < 0.001) continue;
                    const double v = num[r] / den[r];
                    if ((float)v <= kEmpty) continue;
                    sum[r] += v;
                    cnt[r] += 1;
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < RP_ROWS; r++) cnt[r] += plain_cnt;
    reproj_store(a, sum, cnt, (double*)win, y0, x, out);
}

// The same without staged columns, for references so far from the projection
// that those of a single sample do not fit the LDS (lists that are not in the
// order of the tilts: ten references, one of them some 80 degrees from a steep
// projection, spread 64 columns over more than 480).  Every value is looked at for
// being empty.
__global__ __launch_bounds__(64 * RP_WAVES) void k_reproj_far(const float* __restrict__ projs,
                                                              ReprojArgs a, float* __restrict__ out)
{
#pragma clang fp contract(off)
    __shared__ double sums[RP_SUMS / sizeof(double)];
    const int x = blockIdx.x * 64 + (threadIdx.x & 63), wave = threadIdx.x >> 6;
    const int y0 = blockIdx.y * RP_ROWS;
    const double fc = a.ray_cos, fs = a.ray_sin;
    const double cx = a.proj_x * 0.5;
    const int last = a.proj_x - 1;
    const double xp = x + 0.5 - a.proj_x * 0.5;
    const double tx = a.vol_x * 0.5 + a.ray * 0.5 * fs + xp / fc;
    const double tz = a.vol_z * 0.5 - a.ray * 0.5 * fc;
    double sum[RP_ROWS];
    int cnt[RP_ROWS];
#pragma unroll
    for (int r = 0; r < RP_ROWS; r++) {
        sum[r] = 0.0;
        cnt[r] = 0;
    }
    const int per = (a.ray + RP_WAVES - 1) / RP_WAVES;
    const int ia = wave * per, ib = min(ia + per, a.ray);
    for (int i = ia; i < ib; i++) {
        const double px = tx - i * fs;
        const double pz = tz + i * fc;
        if (px < 0 || px >= a.vol_x || pz < 0 || pz >= a.vol_z) continue;
        const double fx = (int)px + 0.5 - a.vol_x * 0.5;
        const double fz = (int)pz + 0.5 - a.vol_z * 0.5;
        double num[RP_ROWS], den[RP_ROWS];
#pragma unroll
        for (int r = 0; r < RP_ROWS; r++) num[r] = den[r] = 0.0;
        for (int k = 0; k < a.n_range; k++) {
            const double u = fx * a.cos_t[k] + fz * a.sin_t[k] + cx;
            if (u < 0 || u > last) continue;
            const float* img = projs + (size_t)(a.first + k) * a.proj_y * a.proj_x + (int)u;
#pragma unroll
            for (int r = 0; r < RP_ROWS; r++) {
                const float v = img[(size_t)min(y0 + r, a.proj_y - 1) * a.proj_x];
                if (v < kEmpty) continue;
                num[r] += v * a.cos_t[k] * a.weight[k];
                den[r] += a.weight[k];
            }
        }
#pragma unroll
        for (int r = 0; r < RP_ROWS; r++) {
            if (den[r] < 0.001) continue;
            const double v = num[r] / den[r];
            if ((float)v <= kEmpty) continue;
            sum[r] += v;
            cnt[r] += 1;
        }
    }
    reproj_store(a, sum, cnt, sums, y0, x, out);
}

// Columns that a segment of n samples reaches at most, over the tilts: 64
// rays a / cos a apart seen at cos t, and the drift of the ray.
static double reach(const ReprojArgs& a, int n)
{
    double w = 0.0;
    for (int k = 0; k < a.n_range; k++)
        w = std::max(w, 63.0 * std::fabs(a.cos_t[k] / a.ray_cos) +
                            n * std::fabs(a.ray_cos * a.sin_t[k] - a.ray_sin * a.cos_t[k]));
    return w + 8.0;
}

template <int N>
static void launch_n(const ReprojArgs& a, size_t shm, const float* projs, float* out, hipStream_t s)
{
    if constexpr (N > 1) {
        if (a.n_range < N) return launch_n<N - 1>(a, shm, projs, out, s);
    }
    // more than 64 KiB of dynamic LDS is asked for once per device
    static std::atomic<unsigned long long> done{0};
    int dev = -1;
    const bool known = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64;
    if (shm > 64 * 1024 && !(known && (done.load(std::memory_order_relaxed) >> dev & 1))) {
        if (hipFuncSetAttribute((const void*)k_reproj<N>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, RP_LDS_MAX) == hipSuccess) {
            if (known) done.fetch_or(1ull << dev, std::memory_order_relaxed);
        } else {
            (void)hipGetLastError();   // the launch reports it
        }
    }
    hipLaunchKernelGGL(k_reproj<N>, dim3((a.proj_x + 63) / 64, (a.proj_y + RP_ROWS - 1) / RP_ROWS),
                       dim3(64 * RP_WAVES), shm, s, projs, a, out);
}

void launch_reproj(const ReprojArgs& args, const float* projs, float* out, hipStream_t s)
{
    ReprojArgs a = args;
    const int entry = RP_ROWS * (int)sizeof(float) * a.n_range;
    auto bytes = [&](int n) { return (size_t)(std::min(reach(a, n), (double)a.proj_x) + 1.0) * entry; };
    if (bytes(1) > (size_t)RP_LDS_MAX) {
        hipLaunchKernelGGL(k_reproj_far, dim3((a.proj_x + 63) / 64, (a.proj_y + RP_ROWS - 1) / RP_ROWS),
                           dim3(64 * RP_WAVES), 0, s, projs, a, out);
        return;
    }
    // the longest equal segments that fit; a lone reference far from a steep
    // projection spreads 64 columns over thousands and takes more LDS
    const size_t limit = bytes(1) <= (size_t)RP_LDS ? RP_LDS : RP_LDS_MAX;
    int n_seg = 1;
    while (n_seg < a.ray && bytes((a.ray + n_seg - 1) / n_seg) > limit) n_seg++;
    a.seg = std::max(1, (a.ray + n_seg - 1) / n_seg);
    a.width = (int)(bytes(a.seg) / entry);
    const size_t shm = std::max((size_t)a.width * entry, (size_t)RP_SUMS);
    launch_n<REPROJ_MAX_TILTS>(a, shm, projs, out, s);
}

}  // namespace atr
