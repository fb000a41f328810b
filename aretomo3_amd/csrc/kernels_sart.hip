// kernels_sart.hip -- pre-stage, weighting, SART back-projection and the
// volume fill/output kernels (gfx950); the forward projection + difference
// is in kernels_fp.hip.
//
// Data layout in HBM (one series):
//   d_aligned [N][aln_y][aln_x]      pre-stage output, -1e30 where empty
//   d_sino    [VolY][N][stride]      weighted projections, sinogram-major:
//                                    the sinogram of slice y is contiguous
//   d_diff    [VolY][max_subset][stride]  SART residual of the current subset
//   d_vol     [VolY][VolZ][VolX]     SART state, x fastest (XZY, unflipped)
#include <atomic>
#include <climits>

#include "atr_internal.h"
#include "storage.h"
#include "work_queue.h"

namespace atr {

// ------------------------------------------------------------------------
// Pre-stage: Correct/GCorrPatchShift.cu:58-100 (global + local shift,
// tilt-axis rotation, nearest neighbour, -1e30 outside the raw image),
// geometry in FP64 with contraction off so that the rounding of every
// coordinate is the rounding of the FP64 restatement.  A wave owns 64 columns
// x 32 rows (16 with patches) of one aligned image and walks down them: near a tilt axis
// of 90 degrees its lanes read 64 raw rows, and the following rows then find
// their samples in the lines already fetched.  (One row per workgroup moved
// 1.4 TB/s: 0.364 ms for 61 images of 1024^2 at 85 degrees, now 0.286; 0.60 ms at
// 0 degrees for 61 of 2048^2, now 0.37.)  Eight rows are loaded at a time.  Each
// workgroup writes the (sum, count) of its non-empty pixels for the fill mean.
//
// PS_LOCAL_FAST: the local shift is the mean of the good patches' shifts
// weighted by exp(-100 d_p^2), d_p the distance to patch p in image sizes.  The
// part of the exponent that is quadratic in the pixel's position is the same
// for every patch and cancels in the mean; what is left is linear, so a
// weight is U_p(x) V_p(y): one exponential per patch and column, one per patch
// and row (in LDS), and per pixel and patch a product and three FMAs instead
// of an FP64 exponential (35.7 -> 5.6 ms for 41 images of 4096^2 with 25
// patches).  The relative error of a weight is about |exponent| 2^-53, as it
// was.  PS_LOCAL evaluates the weights as written, for patches so far from
// the image that the factors or the weights themselves could leave the range
// of a double (ps_local_fast on the host).
// ------------------------------------------------------------------------
enum { PS_GLOBAL = 0, PS_LOCAL_FAST = 1, PS_LOCAL = 2 };
constexpr int PS_CHUNK = 32;   // patches whose row factors are in LDS at once

template <int MODE>
__global__ __launch_bounds__(256) void k_prestage(const float* __restrict__ in, size_t tilt_stride,
                                                  size_t row_stride, int in_x, int in_y,
                                                  const double2* __restrict__ axis_cs,
                                                  const float2* __restrict__ shifts,
                                                  const float* __restrict__ local, int n_patches,
                                                  float* __restrict__ out, int out_x, int out_y,
                                                  double2* __restrict__ block_stats)
{
#pragma clang fp contract(off)
    constexpr int R = ps_rows(MODE != PS_GLOBAL);
    extern __shared__ float s_patch[];
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y0 = blockIdx.y * R, t = blockIdx.z;
    const int n_rows = min(R, out_y - y0);
    const float* lp = MODE == PS_GLOBAL ? nullptr : local + (size_t)t * 5 * n_patches;
    const double ca = axis_cs[t].x, sa = axis_cs[t].y;
    const double sx = (double)shifts[t].x + in_x * 0.5;
    const double sy = (double)shifts[t].y + in_y * 0.5;
    const double xc = x + 0.5 - out_x * 0.5;
    const float* src = in + (size_t)t * tilt_stride;
    float* dst = out + ((size_t)t * out_y + y0) * out_x + x;
    double sum = 0.0;
    int cnt = 0;
    // the raw pixel nearest to (xr, yr): loaded from a clamped position, and
    // used (empty outside the image) once the group's loads are on their way
    auto fetch = [&](double xr, double yr, bool& inside) {
        xr += sx;
        yr += sy;
        const int ix = (int)(xr + 0.5);
        const int iy = (int)(yr + 0.5);
        inside = ix >= 0 && ix < in_x && iy >= 0 && iy < in_y;
        return src[(size_t)min(max(iy, 0), in_y - 1) * row_stride + min(max(ix, 0), in_x - 1)];
    };
    auto store = [&](int r, float v, bool inside) {
        if (!inside) v = kSentinel;
        if (!(v < kEmpty)) {
            sum += v;
            cnt += 1;
        }
        dst[(size_t)r * out_x] = v;
    };
    // G rows from row r0 on (those below the image are loaded and not stored)
    constexpr int G = 8;
    auto rows = [&](int r0, auto position) {
        float v[G];
        bool inside[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            double xr, yr;
            position(r0 + g, xr, yr);
            v[g] = fetch(xr, yr, inside[g]);
        }
#pragma unroll
        for (int g = 0; g < G; g++)
            if (r0 + g < n_rows) store(r0 + g, v[g], inside[g]);
    };
    if constexpr (MODE == PS_LOCAL_FAST) {
        double* v_row = (double*)s_patch;            // [PS_CHUNK][R]
        double* par = v_row + PS_CHUNK * R;          // per patch: a, shift x, y
        double wx[R], wy[R], sw[R];
#pragma unroll
        for (int r = 0; r < R; r++) wx[r] = wy[r] = sw[r] = 0.0;
        int used = 0;
        for (int p0 = 0; p0 < n_patches; p0 += PS_CHUNK) {
            const int np = min(PS_CHUNK, n_patches - p0);
            __syncthreads();
            for (int i = threadIdx.x; i < np * R; i += blockDim.x) {
                const int q = i / R, r = i - q * R;
                const bool good = !(lp[4 * n_patches + p0 + q] < 0.9f);
                // centre over image size squared, times 200
                const double cx = lp[p0 + q], cy = lp[n_patches + p0 + q];
                const double gx = 200.0 * cx / ((double)in_x * in_x);
                const double gy = 200.0 * cy / ((double)in_y * in_y);
                const double yc = (y0 + r) + 0.5 - out_y * 0.5;
                const double e = (gy * ca - gx * sa) * yc - 0.5 * (gx * cx + gy * cy);
                v_row[i] = good ? exp(e) : 0.0;
                if (r == 0) {
                    par[3 * q] = good ? gx * ca + gy * sa : 0.0;
                    par[3 * q + 1] = (double)lp[2 * n_patches + p0 + q];
                    par[3 * q + 2] = (double)lp[3 * n_patches + p0 + q];
                }
            }
            __syncthreads();
            for (int q = 0; q < np; q++) {
                if (lp[4 * n_patches + p0 + q] < 0.9f) continue;
                used += 1;
                const double u = exp(par[3 * q] * xc);
                const double px = par[3 * q + 1], py = par[3 * q + 2];
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const double w = u * v_row[q * R + r];
                    sw[r] += w;
                    wx[r] = fma(px, w, wx[r]);
                    wy[r] = fma(py, w, wy[r]);
                }
            }
        }
        if (x < out_x) {
#pragma unroll
            for (int r0 = 0; r0 < R; r0 += G)
                if (r0 < n_rows)
                    rows(r0, [&](int r, double& xr, double& yr) {
                        const double yc = (y0 + r) + 0.5 - out_y * 0.5;
                        xr = xc * ca - yc * sa;
                        yr = xc * sa + yc * ca;
                        if (used > 0) {
                            const double inv = 1.0 / sw[r];
                            xr += wx[r] * inv;
                            yr += wy[r] * inv;
                        }
                    });
        }
    } else {
        if (MODE == PS_LOCAL) {
            for (int i = threadIdx.x; i < 5 * n_patches; i += blockDim.x) s_patch[i] = lp[i];
            __syncthreads();
        }
        if (x < out_x) {
            for (int r0 = 0; r0 < n_rows; r0 += G)
                rows(r0, [&](int r, double& xr, double& yr) {
                    const double yc = (y0 + r) + 0.5 - out_y * 0.5;
                    xr = xc * ca - yc * sa;
                    yr = xc * sa + yc * ca;
                    if (MODE == PS_LOCAL) {
                        // Correct/GCorrPatchShift.cu:18-48: Gaussian-weighted mean
                        // of the good patches' shifts (good >= 0.9); no weight ->
                        // no shift
                        const float *pcx = s_patch, *pcy = s_patch + n_patches;
                        const float *psx = s_patch + 2 * n_patches, *psy = s_patch + 3 * n_patches;
                        const float* pgood = s_patch + 4 * n_patches;
                        double wx = 0.0, wy = 0.0, sw = 0.0;
                        int used = 0;
                        for (int q = 0; q < n_patches; q++) {
                            if (pgood[q] < 0.9f) continue;
                            double dx = (xr - (double)pcx[q]) / in_x;
                            double dy = (yr - (double)pcy[q]) / in_y;
                            double w = exp(-100.0 * (dx * dx + dy * dy));
                            wx += (double)psx[q] * w;
                            wy += (double)psy[q] * w;
                            sw += w;
                            used += 1;
                        }
                        if (used > 0 && sw > 0) {
                            xr += wx / sw;
                            yr += wy / sw;
                        }
                    }
                });
        }
    }
    // fixed-order block reduction (deterministic)
    __shared__ double s_sum[256];
    __shared__ int s_cnt[256];
    s_sum[threadIdx.x] = sum;
    s_cnt[threadIdx.x] = cnt;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o && threadIdx.x + o < blockDim.x) {
            s_sum[threadIdx.x] += s_sum[threadIdx.x + o];
            s_cnt[threadIdx.x] += s_cnt[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        block_stats[((size_t)t * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] =
            make_double2(s_sum[0], (double)s_cnt[0]);
}

// Per-tilt fill statistics: sum of the workgroups' partials in a fixed order.
__global__ __launch_bounds__(256) void k_tilt_stats(const double2* __restrict__ block_stats, int blocks,
                                                    double2* __restrict__ tilt_stats)
{
    const int t = blockIdx.x;
    double sum = 0.0, cnt = 0.0;
    for (int i = threadIdx.x; i < blocks; i += blockDim.x) {
        double2 r = block_stats[(size_t)t * blocks + i];
        sum += r.x;
        cnt += r.y;
    }
    __shared__ double s_sum[256], s_cnt[256];
    s_sum[threadIdx.x] = sum;
    s_cnt[threadIdx.x] = cnt;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            s_sum[threadIdx.x] += s_sum[threadIdx.x + o];
            s_cnt[threadIdx.x] += s_cnt[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) tilt_stats[t] = make_double2(s_sum[0], s_cnt[0]);
}

// Value of aligned pixel i of tilt t after MaUtil/GFillEmpty2D.cu:60-88:
// an empty pixel follows the random chain (<= 100 hops) to the first
// non-empty pixel, else takes the tilt mean.  Reads only the unfilled
// image, so every pixel can be resolved independently.
__device__ __forceinline__ float filled_value(const float* __restrict__ img, int i,
                                              const int* __restrict__ table, float mean)
{
    float v = img[i];
    if (!(v < kEmpty)) return v;
    int next = table[i];
    for (int j = 0; j < 100; j++) {
        float w = img[next];
        if (w < kEmpty) {
            next = table[next];
            continue;
        }
        return w;
    }
    return mean;
}

// ------------------------------------------------------------------------
// Weighting (Recon/GWeightProjs.cu:7-19): s *= cos_t / VolZ, written
// sinogram-major into d_sino, with the pre-stage random fill resolved on the
// fly.  One thread per pixel; grid (x-blocks, tilt, y).
// ------------------------------------------------------------------------
template <typename S>
__global__ __launch_bounds__(256) void k_weight(const float* __restrict__ in, size_t tilt_stride,
                                                size_t row_stride, int fill,
                                                const int* __restrict__ table,
                                                const double2* __restrict__ tilt_stats,
                                                const float2* __restrict__ cs, int n, int proj,
                                                int vol_z, S* __restrict__ sino, int stride,
                                                int* __restrict__ sflag)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int t = blockIdx.y, y = blockIdx.z;
    if (x >= stride) return;
    S* dst = sino + ((size_t)y * n + t) * stride;
    if (x >= proj) {
        st<S>(dst + x, 0.0f);
        return;
    }
    const float w = cs[t].x / (float)vol_z;
    const float* img = in + (size_t)t * tilt_stride;
    float v;
    if (fill) {
        double2 ts = tilt_stats[t];
        float mean = ts.y > 0 ? (float)(ts.x / ts.y) : 0.0f;
        v = filled_value(img, (int)(y * row_stride + x), table, mean);
    } else {
        v = img[(size_t)y * row_stride + x];
    }
    v *= w;
    if (v <= kEmpty) atomicOr(sflag + y, 1);
    st<S>(dst + x, v);
}

// ------------------------------------------------------------------------
// SART back-projection (Recon/GBackProj.cu:12-60).
//
// Workgroup = BP_TX x (BP_WAVES TZ) voxels of one slice (64 x 64 at TZ = 16),
// lane = x, wave = a quarter of the rows, each thread walks TZ z-rows.  For
// each chunk of CH tilts the part of every sinogram row that the tile can
// reach (at most |cos| 63 + |sin| 63 samples and guards: 96 at TZ = 16) is
// staged in LDS as pairs (A_i, d_i), d_i = q_{i+1} - q_i, A_i = q_i -
// (i - 1/2) d_i, so that a voxel's value is the one FMA A_i + v d_i at
// v = u - 1/2, u its coordinate in the window.  A square tile reaches the
// fewest samples for its voxels: 0.023 pairs are staged per update, against
// 0.070 for 256 x 16 voxels.
//
// The cell index costs two instructions: v + (2^23 + window base) rounds v to
// the nearest integer, which is floor(u), into the low bits of the float
// (a tie, u an integer, may take the cell below: both give the same value),
// and a 16-bit shift makes those bits the byte address.  Both, like FMAs and
// adds on vector registers, are instructions of which the SIMD issues two at
// a time, from two waves; conversions, 32-bit left shifts and anything with a
// scalar operand issue one at a time (measured: 2.3 and 4 cycles per wave
// instruction at four waves per SIMD).  All operands of an update are
// therefore vector registers, and its five instructions take 11.5 cycles,
// against 14.5 with a scalar slope, a conversion and a shift-add.
//
// Inclusion comes from the FP64 interval tables: tiles the host classified as
// fully inside skip all per-lane tests and count per tile; partial tiles test
// x against the (tilt, z) interval.  Sums and counts are FP32/int per voxel,
// in tilt order, as the reference.  What a wave needs per tilt (coordinate of
// its first voxel, cos, sin, class) is put into LDS with the rows and read
// one tilt ahead, so no scalar-load latency stands between two tilts.
//
// BF16 storage runs SART on wide tiles (256 x TZ, waves side by side in x), with
// coordinates rounded relative to the tile's first voxel, truncated and scaled
// as they always were there: the differences are stored in BF16 after every
// step, so a coordinate rounded otherwise, however little, moves some of them
// by a whole unit of 2^-8, and single voxels by 1e-3 of the volume's rms.
//
// 1024^2 x 256, 12 to 13 tilts: 0.55 ms a launch (0.895 with 256 x 16 voxel
// tiles, scalar operands and a conversion per update); 4.0 TB/s of the 4.9 a
// large copy reaches.  WBP grid of 512^2 x 128, 41 tilts: 0.71 ms (1.29).  What
// bounds it is the LDS (one 8-byte read per update: 9 cycles per SIMD) beside
// the 11.5 issue cycles of an update; 5 (WBP: 6) waves per SIMD hide the
// staging loads and the barrier.
// ------------------------------------------------------------------------
template <int TZ, int CH, int KIND>
struct BpLds {
    float2 pairs[CH * bp_win(TZ, KIND)];
    // per wave and tilt: u - w0 - 1/2 at the wave's first voxel (wide: u - w0
    // at the tile's), scaled cos and sin, class; one spare entry, read ahead of
    // the last tilt
    float4 ent[BP_WAVES][CH + 1];
};

// Byte address of the pair that v (plus the 2^23 of cm) falls into.
// Wide tiles: v is the coordinate itself, truncated, and cm carries the bits of
// the window's byte offset.
template <bool WIDE>
__device__ __forceinline__ unsigned bp_addr(float v, float cm)
{
    if constexpr (WIDE) return 8 * (int)v + __float_as_int(cm);
    unsigned a;
    asm("v_lshlrev_b16 %0, 3, %1" : "=v"(a) : "v"(v + cm));
    return a;
}

// v0 + k ss with k as the instruction's literal (a constant in a scalar
// register would halve the issue rate).
template <int K>
__device__ __forceinline__ float bp_coord(float ss, float v0)
{
    if constexpr (K == 0) return v0;
    if constexpr (K == 1) return v0 + ss;
    float r;
    asm("v_fmamk_f32 %0, %1, %2, %3"
        : "=v"(r)
        : "v"(ss), "i"(__builtin_bit_cast(int, (float)K)), "v"(v0));
    return r;
}

// Rows K0 .. K0 + 7 of a tilt that every voxel uses: the eight LDS reads go
// out before the first value is needed.
template <int K0, int TZ, bool WIDE>
__device__ __forceinline__ void bp_full8(const char* pairs, float ss, float v0, float cm,
                                         float (&acc)[TZ])
{
    float v[8];
    float2 pr[8];
    v[0] = bp_coord<K0>(ss, v0);
    v[1] = bp_coord<K0 + 1>(ss, v0);
    v[2] = bp_coord<K0 + 2>(ss, v0);
    v[3] = bp_coord<K0 + 3>(ss, v0);
    v[4] = bp_coord<K0 + 4>(ss, v0);
    v[5] = bp_coord<K0 + 5>(ss, v0);
    v[6] = bp_coord<K0 + 6>(ss, v0);
    v[7] = bp_coord<K0 + 7>(ss, v0);
#pragma unroll
    for (int k = 0; k < 8; k++) pr[k] = *(const float2*)(pairs + bp_addr<WIDE>(v[k], cm));
#pragma unroll
    for (int k = 0; k < 8; k++) acc[K0 + k] += fmaf(v[k], pr[k].y, pr[k].x);
}

// The x-intervals of eight rows of one tilt, one scalar load.
struct BpRows8 {
    int2 r[8];
};

// One tile.  The caller puts a barrier between two tiles of a workgroup.
//
// SENT: the slice's sinogram rows may hold empty samples.  The staged pair is
// then (q_i, d_i) and the value q + fract(u) d, whose sentinel test must see
// the exact -1e30 scale.
template <typename S, int TZ, int CH, int KIND, bool SENT>
__device__ __forceinline__ void bp_tile_body(cptr<BpArgs> A, BpLds<TZ, CH, KIND>& lds, int xt,
                                             int zt, int y)
{
    constexpr bool WBP = KIND == BP_GRID, WIDE = KIND == BP_WIDE;
    constexpr int WIN = bp_win(TZ, KIND);
    // waves side by side in x and in z
    constexpr int WX = bp_wx(KIND), WZ = BP_WAVES / WX;
    const int rows_per_slice = A->rows_per_slice, stride = A->stride, proj = A->proj;
    const int n_list = A->n_list;
    const int vol_x = A->vol_x, vol_z = A->vol_z;
    const float relax = A->relax;
    const int positivity = A->positivity;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int xq = xt * WX + wave % WX, zq = zt * WZ + wave / WX, z0 = zq * TZ;
    const bool live = z0 < vol_z && xq * BP_TX < vol_x;
    const int x = xq * BP_TX + lane;
    const int xc = min(x, vol_x - 1);
    // the slice and its sinogram rows as buffers: a row offset is a scalar, a
    // column the lane's fixed byte offset
    const gptr<float> vslice = as_gptr(A->vol) + (size_t)y * vol_z * vol_x;
    const __amdgpu_buffer_rsrc_t vres =
        buffer_of((const void*)vslice, (size_t)vol_z * vol_x * sizeof(float));
    const int row_bytes = vol_x * (int)sizeof(float);
    const gptr<const S> base = (gptr<const S>)A->sino + (size_t)y * rows_per_slice * stride;
    const __amdgpu_buffer_rsrc_t sres =
        buffer_of((const void*)base, (size_t)rows_per_slice * stride * sizeof(S));
    // window starts are those of the workgroup's tile (the same in the
    // entries of all its waves); coordinates and classes are the wave's
    const size_t entries = ((size_t)zq * (A->n_xtiles * WX) + xq) * n_list;
    const gptr<const int2> etab = as_gptr(A->tiles) + entries;

    float vold[TZ];
    float acc[TZ];
    // counts of the partial tiles, two 16-bit counts to a register
    unsigned cnt[TZ / 2];
#pragma unroll
    for (int k = 0; k < TZ; k++) acc[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < TZ / 2; k++) cnt[k] = 0;
    int full_cnt = 0;
    bool partial = false;
    const float xf = (float)(xc - xt * WX * BP_TX);   // offset from the tile's first voxel

    for (int c0 = 0; c0 < n_list; c0 += CH) {
        const int nc = min(CH, n_list - c0);
        if (c0 > 0) __syncthreads();
        // ---- stage: wave w takes the ROUNDS tilts from w ROUNDS on.  Pair i
        // of a row is (q(g), q(g+1) - q(g)) at g = w0 + i, where q is the row
        // extended linearly beyond its ends: q(g) = p[ga] + (g - ga)
        // (p[ga+1] - p[ga]), ga = clamp(g, 0, P-2).  Inside [0, P-2] that is
        // the plain pair; at g = -1 it extrapolates, so a coordinate that FP32
        // rounding puts just below 0 still interpolates the first sample.
        // Pairs further out are only read by voxels the exact intervals
        // exclude.  Each 64 pairs of a tilt take one wave instruction, the U
        // others share one with those of GU - 1 more tilts.  Past the list's
        // end the tables go on (into the next list, or their padding): what is
        // staged for those slots is not read.  All loads are issued before a
        // pair is formed, on every path alike (wide tiles, whose windows are
        // longer: two tilts at a time). ----
        constexpr int ROUNDS = CH / BP_WAVES, RND = WIDE ? 2 : ROUNDS;
        constexpr int MF = WIN / 64, U = WIN % 64, GU = U > 0 ? 64 / U : 1;
        constexpr int UP = U > 0 ? (RND + GU - 1) / GU : 0, NP = RND * MF + UP;
        struct WindowStarts {
            int2 e[RND];
        };
        struct Tilts {
            BpTilt t[RND];
        };
#pragma unroll
        for (int h = 0; h < ROUNDS; h += RND) {
            const int jw = wave * ROUNDS + h;
            const WindowStarts ws = ldc((cptr<WindowStarts>)(as_cptr(A->tiles) + entries + c0 + jw));
            const Tilts tl = ldc((cptr<Tilts>)(as_cptr(A->list) + c0 + jw));
            float2 pv[NP];
            int ga[NP], w0v[NP], slot[NP];
#pragma unroll
            for (int q = 0; q < NP; q++) {
                int w0, voff, soff = 0;
                if (q < RND * MF) {
                    const int r = q / MF, i = lane + q % MF * 64;
                    w0 = ws.e[r].x >> 2;
                    slot[q] = (jw + r) * WIN + i;
                    ga[q] = min(max(w0 + i, 0), proj - 2);
                    voff = ga[q] * (int)sizeof(S);
                    soff = tl.t[r].row * stride * (int)sizeof(S);
                } else {
                    // lanes U s .. U s + U - 1: the upper pairs of tilt
                    // (q - RND MF) GU + s (the last one again past the wave's)
                    const int s = lane / (U > 0 ? U : 64), i = MF * 64 + lane % (U > 0 ? U : 64);
                    int row = 0, r = 0;
                    w0 = 0;
#pragma unroll
                    for (int g = 0; g < GU; g++) {
                        const int qq = min((q - RND * MF) * GU + g, RND - 1);
                        if (g == 0 || s >= g) {
                            w0 = ws.e[qq].x >> 2;
                            row = tl.t[qq].row;
                            r = qq;
                        }
                    }
                    slot[q] = (jw + r) * WIN + i;
                    ga[q] = min(max(w0 + i, 0), proj - 2);
                    voff = (row * stride + ga[q]) * (int)sizeof(S);
                }
                w0v[q] = w0;
                pv[q] = ldb2<S>(sres, voff, soff);
            }
#pragma unroll
            for (int q = 0; q < NP; q++) {
                float p = pv[q].x, r = pv[q].y;
                if constexpr (SENT && !std::is_same<S, float>::value) {
                    // narrow storage cannot hold -1e30: widen its empty marks
                    // (a slice without them has nothing to widen)
                    const float thr = empty_threshold<S>();
                    if (p <= thr) p = kSentinel;
                    if (r <= thr) r = kSentinel;
                }
                const float d = r - p;
                // SENT: the extended value; else that minus (i - 1/2) d (wide:
                // i d)
                const int i = q < RND * MF ? lane + q % MF * 64 : MF * 64 + lane % (U > 0 ? U : 64);
                const float gi = SENT ? (float)(w0v[q] + i - ga[q])
                                      : (float)(w0v[q] - ga[q]) + (WIDE ? 0.0f : 0.5f);
                lds.pairs[slot[q]] = make_float2(fmaf(gi, d, p), d);
            }
        }
        if (lane < nc) {
            const int2 e = ldgo(etab + c0 + lane);
            const BpTilt bt = ldgo(as_gptr(A->list) + c0 + lane);
            lds.ent[wave][lane] = make_float4(__int_as_float(e.y), bt.c, bt.s,
                                              __int_as_float(e.x & 3));
        }
        __syncthreads();
        if (!live) continue;
        // the voxels this thread updates, loaded beside the last chunk's
        // sums (the WBP grid is written, not updated)
        if (!WBP && c0 + CH >= n_list) {
            int zo = z0;
            asm volatile("" : "+s"(zo));   // the row offsets are formed here, not kept in registers
#pragma unroll
            for (int k = 0; k < TZ; k++)
                vold[k] = ldb<float>(vres, xc * (int)sizeof(float), min(zo + k, vol_z - 1) * row_bytes);
        }
        // ---- accumulate ----
        const char* pairs = (const char*)lds.pairs;
        float4 next = lds.ent[wave][0];
        // wide: the byte offset of the tilt's window, as an integer
        float cm = WIDE ? 0.0f : 8388608.0f;
        auto next_window = [&] {
            if (WIDE) cm = __int_as_float(__float_as_int(cm) + WIN * 8);
            else cm += (float)WIN;
        };
        for (int j = 0; j < nc;) {
            float4 e;
            int cls;
            // the tilts that every voxel uses run in a loop of their own: as
            // one branch of a common loop, all sums were copied after a tilt
            for (;;) {
                e = next;
                next = lds.ent[wave][j + 1];
                cls = __builtin_amdgcn_readfirstlane(__float_as_int(e.w));
                if (SENT || cls != 1) break;
                full_cnt += 1;
                const float v0 = fmaf(xf, e.y, e.x);
                bp_full8<0, TZ, WIDE>(pairs, e.z, v0, cm, acc);
                if constexpr (TZ > 8) bp_full8<8, TZ, WIDE>(pairs, e.z, v0, cm, acc);
                next_window();
                if (++j >= nc) break;
            }
            if (j >= nc) break;
            const float ss = e.z;
            const float v0 = fmaf(xf, e.y, e.x);
            const int jp = j++;
            const float cp = cm;
            next_window();
            if (cls == 0) continue;
            partial = true;
            const cptr<int2> lh = as_cptr(A->lohi) +
                                  (size_t)ldc(as_cptr(A->list) + c0 + jp).tilt * A->lohi_stride + z0;
#pragma unroll
            for (int k0 = 0; k0 < TZ; k0 += 8) {
                const BpRows8 rows = ldc((cptr<BpRows8>)(lh + k0));
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    const int k = k0 + m;
                    const float v = fmaf((float)k, ss, v0);
                    float val;
                    bool in = (x >= rows.r[m].x) & (x <= rows.r[m].y);
                    if (SENT) {
                        const float u = WIDE ? v : v + 0.5f;
                        const float2 pr = lds.pairs[jp * WIN + (int)u];
                        val = fmaf(__builtin_amdgcn_fractf(u), pr.y, pr.x);
                        in = in & !(val <= kEmpty);
                    } else {
                        const float2 pr = *(const float2*)(pairs + bp_addr<WIDE>(v, cp));
                        val = fmaf(v, pr.y, pr.x);
                    }
                    acc[k] += in ? val : 0.0f;
                    cnt[k / 2] += in ? (k % 2 ? 0x10000u : 1u) : 0u;
                }
            }
        }
    }
    if (!live || x >= vol_x) return;
    const int n_rows = min(TZ, vol_z - z0);
    const int voff = x * (int)sizeof(float);
    bool wrote_sent = false;
    // one row: its sum, the reciprocal of its count (with the relaxation)
    auto write = [&](int k, float scale, bool any) {
        const int so = (z0 + k) * row_bytes;
        if (WBP) {
            // mean over the tilts used, 0 when none (GBackProjWbp.cu:48-52)
            stb(vres, any ? acc[k] * scale : 0.0f, voff, so);
        } else {
            // v = relax * sum / count + v, positivity, sentinel (GBackProj.cu:50-59)
            float v = WIDE ? fmaf(relax * acc[k], scale, vold[k]) : fmaf(acc[k], scale, vold[k]);
            const bool empty = !(v > kEmpty);
            v = empty ? kSentinel : (positivity ? fmaxf(v, 0.0f) : v);
            if (any) {
                stb(vres, v, voff, so);
                wrote_sent |= empty;
            }
        }
    };
    // every voxel of a wave without partial tiles used the same tilts
    const float num = WBP || WIDE ? 1.0f : relax;
    const float one = num * __builtin_amdgcn_rcpf((float)full_cnt);
    auto rows = [&](auto all) {
#pragma unroll
        for (int k = 0; k < TZ; k++) {
            if (!decltype(all)::value && k >= n_rows) break;
            if (!partial) {
                write(k, one, full_cnt > 0);
            } else {
                const int count = full_cnt + (int)((cnt[k / 2] >> (k % 2 * 16)) & 0xffffu);
                write(k, num * __builtin_amdgcn_rcpf((float)count), count > 0);
            }
        }
    };
    if (!WBP && !partial && full_cnt == 0) return;
    if (!partial && n_rows == TZ) rows(std::true_type{});
    else rows(std::false_type{});
    if (!WBP && wrote_sent) atomicOr(A->vflag + y, 1);
}

template <typename S, int TZ, int CH, int KIND>
__device__ __forceinline__ void bp_tile(cptr<BpArgs> A, BpLds<TZ, CH, KIND>& lds, int xt, int zt,
                                        int y)
{
    const cptr<int> sflag = as_cptr(A->sflag);
    if (sflag != nullptr && sflag[y] != 0)
        bp_tile_body<S, TZ, CH, KIND, true>(A, lds, xt, zt, y);
    else
        bp_tile_body<S, TZ, CH, KIND, false>(A, lds, xt, zt, y);
}

// SART tiles of a storage type (bp_kind_of on the host).
template <typename S>
constexpr int bp_kind()
{
    return std::is_same<S, bf16_t>::value ? BP_WIDE : BP_SQUARE;
}

// n_y > 0: grid (8 x-tiles, z-tiles, slices / 8), n_y slices.  Workgroups go
// to the eight XCDs in turn, so all tiles of a slice run on one XCD, whose L2
// holds the slice's sinogram.  n_y = 0: grid (x-tiles, z-tiles, slices), for
// few slices, whose tiles spread over the XCDs (bp_grid).
template <typename S, int TZ, int CH>
__global__ __launch_bounds__(BP_THREADS, 5) void k_back_proj(const BpArgs* __restrict__ a, int n_y)
{
    constexpr int KIND = bp_kind<S>();
    __shared__ BpLds<TZ, CH, KIND> lds;
    const int per = n_y > 0 ? XCDS : 1;
    const int y = blockIdx.z * per + blockIdx.x % per;
    if (n_y > 0 && y >= n_y) return;
    bp_tile<S, TZ, CH, KIND>(as_cptr(a), lds, blockIdx.x / per, blockIdx.y, y);
}

// WBP back-projection onto the 2x grid (Recon/GBackProjWbp.cu:14-53): the
// same tile machinery, coordinate u = (fx cos + fz sin)/2 + P/2 + 1/2, the
// mean written to the grid buffer.
template <typename S, int TZ>
__global__ __launch_bounds__(BP_THREADS, 6) void k_wbp_grid_bp(const BpArgs* __restrict__ a, int n_y)
{
    __shared__ BpLds<TZ, BP_WBP_CHUNK, BP_GRID> lds;
    const int per = n_y > 0 ? XCDS : 1;
    const int y = blockIdx.z * per + blockIdx.x % per;
    if (n_y > 0 && y >= n_y) return;
    bp_tile<S, TZ, BP_WBP_CHUNK, BP_GRID>(as_cptr(a), lds, blockIdx.x / per, blockIdx.y, y);
}

// Back-projection of many series in persistent launches: blocks take
// (series, slice, run of BP_ITEM_TILES tiles) items from a queue; entries
// are ordered by their first item.  One launch runs one tile shape (0: 16 z rows x 16 tilts
// per stage, 1: 16 x 8, 2: 8 x 16, 3: 8 x 8), so each shape's kernel holds
// only its own code and registers.  Shape 0 takes 97 VGPRs, 4 waves per SIMD
// (k_back_proj<float, 16, 16>: 87, and 5): 16 uneven series spend 300 ms here,
// 250 series by series.
template <typename S, int SHAPE>
__global__ __launch_bounds__(BP_THREADS) void k_back_proj_batch(const BpItem* __restrict__ e, int n_e,
                                                           int total, int* __restrict__ counter)
{
    constexpr int TZ = (SHAPE & 2) ? 8 : 16, CH = (SHAPE & 1) ? 8 : 16;
    constexpr int KIND = bp_kind<S>();
    __shared__ BpLds<TZ, CH, KIND> lds;
    const cptr<BpItem> E = as_cptr(e);
    int s = 0;
    for (int it = publish_item(claim_item(counter)); it < total;) {
        const int ahead = claim_item(counter);
        s = entry_of(E, n_e, it, s);
        const int local = it - E[s].item0;
        const int per_y = E[s].n_items_y;
        const int y = local / per_y, q = local - y * per_y;
        const int nx = E[s].a.n_xtiles, nt = E[s].a.n_ztiles * nx;
        for (int g = 0; g < BP_ITEM_TILES; g++) {
            const int r = q * BP_ITEM_TILES + g;
            if (r >= nt) break;
            const int zt = r / nx, xt = r - zt * nx;
            if (g > 0) __syncthreads();
            bp_tile<S, TZ, CH, KIND>(&E[s].a, lds, xt, zt, y);
        }
        it = publish_item(ahead);
    }
}

// ------------------------------------------------------------------------
// Volume helpers: zero / load the SART state, per-slice fill statistics,
// output with the fill of MaUtil/GFillEmpty2D.cu:60-88 (CTomoSart.cpp:86-89)
// and the z-flip / XYZ layouts of CDoSartRecon.cpp:253-269 and
// DataUtil/CTiltSeries.cpp:286-305.
// ------------------------------------------------------------------------
__global__ void k_fill_zero(float* __restrict__ p, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0.0f;
}

__global__ void k_fill_zero_int(int* __restrict__ p, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// SLICE-layout caller volume -> state, flagging slices that hold empties.
__global__ __launch_bounds__(256) void k_load_volume(const float* __restrict__ in,
                                                     float* __restrict__ vol, int vol_x,
                                                     int vol_z, int* __restrict__ vflag)
{
    const int y = blockIdx.y;
    const size_t n = (size_t)vol_x * vol_z;
    bool any = false;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        float v = in[(size_t)y * n + i];
        vol[(size_t)y * n + i] = v;
        any |= v < kEmpty;
    }
    if (any) atomicOr(vflag + y, 1);
}

// (sum, count) of non-empty voxels of each flagged slice, fixed order.
__global__ __launch_bounds__(256) void k_vol_stats(const float* __restrict__ vol, int vol_x,
                                                   int vol_z, const int* __restrict__ vflag,
                                                   double2* __restrict__ stats)
{
    const int y = blockIdx.x;
    if (vflag[y] == 0) return;
    const size_t n = (size_t)vol_x * vol_z;
    const float* v = vol + (size_t)y * n;
    double sum = 0.0, cnt = 0.0;
    for (size_t i = threadIdx.x; i < n; i += blockDim.x) {
        float a = v[i];
        if (!(a < kEmpty)) {
            sum += a;
            cnt += 1.0;
        }
    }
    __shared__ double s_sum[256], s_cnt[256];
    s_sum[threadIdx.x] = sum;
    s_cnt[threadIdx.x] = cnt;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            s_sum[threadIdx.x] += s_sum[threadIdx.x + o];
            s_cnt[threadIdx.x] += s_cnt[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) stats[y] = make_double2(s_sum[0], s_cnt[0]);
}

__device__ __forceinline__ size_t out_index(int layout, int x, int y, int z, int vol_x,
                                            int vol_y, int vol_z)
{
    switch (layout) {
    case ATR_LAYOUT_XYZ: return ((size_t)z * vol_y + y) * vol_x + x;
    case ATR_LAYOUT_XYZ_NOFLIP: return ((size_t)(vol_z - 1 - z) * vol_y + y) * vol_x + x;
    case ATR_LAYOUT_SLICE: return ((size_t)y * vol_z + z) * vol_x + x;
    default: return ((size_t)y * vol_z + (vol_z - 1 - z)) * vol_x + x;
    }
}

// grid (x-blocks, z, y)
__global__ __launch_bounds__(256) void k_output(const float* __restrict__ vol, int vol_x,
                                                int vol_y, int vol_z, const int* __restrict__ vflag,
                                                const double2* __restrict__ stats,
                                                const int* __restrict__ table, int layout,
                                                float* __restrict__ out)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int z = blockIdx.y, y = blockIdx.z;
    if (x >= vol_x) return;
    const float* slice = vol + (size_t)y * vol_z * vol_x;
    float v = slice[(size_t)z * vol_x + x];
    if (vflag[y] != 0 && v < kEmpty) {
        double2 st2 = stats[y];
        float mean = st2.y > 0 ? (float)(st2.x / st2.y) : 0.0f;
        v = filled_value(slice, z * vol_x + x, table, mean);
    }
    out[out_index(layout, x, y, z, vol_x, vol_y, vol_z)] = v;
}

// Plain streaming copy (16 B per lane, grid-stride, four independent loads
// in flight per lane): the calibration kernel for HBM byte counters and the
// attainable-bandwidth reference.
__global__ __launch_bounds__(256) void k_copy(const float4* __restrict__ src,
                                              float4* __restrict__ dst, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const float4 a = src[i], b = src[i + stride], c = src[i + 2 * stride],
                     d = src[i + 3 * stride];
        dst[i] = a;
        dst[i + stride] = b;
        dst[i + 2 * stride] = c;
        dst[i + 3 * stride] = d;
    }
    for (; i < n; i += stride) dst[i] = src[i];
}

void launch_copy(const void* src, void* dst, size_t bytes, hipStream_t s)
{
    size_t n = bytes / sizeof(float4);
    if (n == 0) return;
    unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_copy, dim3(blocks), dim3(256), 0, s, (const float4*)src, (float4*)dst, n);
}

// ------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------
// Grid of the pre-stage: up to four waves of 64 columns side by side.
static dim3 ps_grid(const Plan& p, int* threads)
{
    *threads = 64 * std::min(4, (p.aln_x + 63) / 64);
    const int rows = ps_rows(p.n_patches > 0);
    return dim3((p.aln_x + *threads - 1) / *threads, (p.aln_y + rows - 1) / rows, p.n);
}

int ps_blocks(const Plan& p)
{
    int threads = 0;
    const dim3 g = ps_grid(p, &threads);
    return (int)(g.x * g.y);
}

template <int MODE>
static void launch_prestage_t(const Plan& p, const float* in, size_t shm, hipStream_t s)
{
    int threads = 0;
    const dim3 grid = ps_grid(p, &threads);
    hipLaunchKernelGGL(k_prestage<MODE>, grid, dim3(threads), shm, s, in, p.in_tilt_stride,
                       p.in_row_stride, p.in_x, p.in_y, (const double2*)p.d_axis_cs,
                       (const float2*)p.d_shifts, p.d_local, p.n_patches, p.d_aligned, p.aln_x,
                       p.aln_y, (double2*)p.d_block_stats);
}

void launch_prestage(const Plan& p, const float* in, hipStream_t s)
{
    if (p.n_patches == 0) launch_prestage_t<PS_GLOBAL>(p, in, 0, s);
    else if (p.local_fast)
        launch_prestage_t<PS_LOCAL_FAST>(p, in, sizeof(double) * PS_CHUNK * (ps_rows(true) + 3), s);
    else launch_prestage_t<PS_LOCAL>(p, in, sizeof(float) * 5 * (size_t)p.n_patches, s);
}

void launch_tilt_stats(const Plan& p, hipStream_t s)
{
    hipLaunchKernelGGL(k_tilt_stats, dim3(p.n), dim3(256), 0, s, (const double2*)p.d_block_stats,
                       ps_blocks(p), (double2*)p.d_tilt_stats);
}

template <typename S>
static void launch_weight_t(const Plan& p, const float* in, hipStream_t s)
{
    const StageSource src0 = stage_source(p, in);
    const float* src = src0.src;
    const size_t ts = src0.tilt_stride, rs = src0.row_stride;
    dim3 grid((p.sino_stride + 255) / 256, p.n, p.vol_y);
    hipLaunchKernelGGL(k_weight<S>, grid, dim3(256), 0, s, src, ts, rs, src0.fill ? 1 : 0,
                       p.d_fill_aln, (const double2*)p.d_tilt_stats, p.d_cs, p.n, p.proj,
                       p.vol_z, (S*)p.d_sino, p.sino_stride, p.d_sflag);
}

void launch_weight_sart(const Plan& p, const float* in, hipStream_t s)
{
    if (p.storage == ATR_STORAGE_F16) launch_weight_t<_Float16>(p, in, s);
    else if (p.storage == ATR_STORAGE_BF16) launch_weight_t<bf16_t>(p, in, s);
    else launch_weight_t<float>(p, in, s);
}

BpArgs bp_args(const Plan& p, const void* sino, int rows, int first, int n_list, float relax,
               bool check_sent)
{
    BpArgs a{};
    a.sino = sino;
    a.rows_per_slice = rows;
    a.stride = p.sino_stride;
    a.proj = p.proj;
    a.list = p.d_lists + first;
    a.n_list = n_list;
    a.lohi = p.d_bp_lohi;
    a.lohi_stride = bp_zpad(p.vol_z);
    const int kind = bp_kind_of(p.storage);
    a.n_ztiles = bp_ztiles(p.vol_z, p.bp_tz, kind);
    a.n_xtiles = bp_xtiles(p.vol_x, kind);
    a.tiles = p.d_bp_tiles + (size_t)a.n_ztiles * BP_WAVES * a.n_xtiles * first;
    a.relax = relax;
    a.positivity = p.positivity;
    a.sflag = check_sent ? p.d_sflag : nullptr;
    a.vol = p.d_vol;
    a.vol_x = p.vol_x;
    a.vol_z = p.vol_z;
    a.vflag = p.d_vflag;
    return a;
}

// Grid of a back-projection; *n_y: its argument.
static dim3 bp_grid(int vol_x, int vol_y, int vol_z, int tz, int kind, int* n_y)
{
    const int nxt = bp_xtiles(vol_x, kind), nzt = bp_ztiles(vol_z, tz, kind);
    if (vol_y < BP_XCD_SLICES) {
        *n_y = 0;
        return dim3(nxt, nzt, vol_y);
    }
    *n_y = vol_y;
    return dim3(XCDS * nxt, nzt, (vol_y + XCDS - 1) / XCDS);
}

template <typename S, int TZ, int CH>
static void launch_bp_v(const Plan& p, int step, hipStream_t s)
{
    int n_y = 0;
    const dim3 grid = bp_grid(p.vol_x, p.vol_y, p.vol_z, TZ, bp_kind<S>(), &n_y);
    hipLaunchKernelGGL((k_back_proj<S, TZ, CH>), grid, dim3(BP_THREADS), 0, s, p.d_bp_args + step,
                       n_y);
}

// Back-projection tile shapes the autotuner chooses from: z rows per thread
// x tilts per LDS stage.
template <typename S>
static void launch_bp_t(const Plan& p, int step, hipStream_t s)
{
    if (p.bp_tz == 8 && p.bp_chunk == 8) launch_bp_v<S, 8, 8>(p, step, s);
    else if (p.bp_tz == 8) launch_bp_v<S, 8, 16>(p, step, s);
    else if (p.bp_chunk == 8) launch_bp_v<S, 16, 8>(p, step, s);
    else launch_bp_v<S, 16, 16>(p, step, s);
}

void launch_bp(const Plan& p, int step, hipStream_t s)
{
    if (p.storage == ATR_STORAGE_F16) launch_bp_t<_Float16>(p, step, s);
    else if (p.storage == ATR_STORAGE_BF16) launch_bp_t<bf16_t>(p, step, s);
    else launch_bp_t<float>(p, step, s);
}

template <typename S>
static void launch_wbp_bp_t(const Plan& p, const BpArgs* a, int ny, hipStream_t s)
{
    int n_y = 0;
    const dim3 grid = bp_grid(2 * p.vol_x, ny, 2 * p.vol_z, p.bp_tz, BP_GRID, &n_y);
    if (p.bp_tz == 8)
        hipLaunchKernelGGL((k_wbp_grid_bp<S, 8>), grid, dim3(BP_THREADS), 0, s, a, n_y);
    else
        hipLaunchKernelGGL((k_wbp_grid_bp<S, 16>), grid, dim3(BP_THREADS), 0, s, a, n_y);
}

void launch_wbp_bp(const Plan& p, int slab, int ny, hipStream_t s)
{
    const BpArgs* a = p.d_bp_args + slab;
    if (p.storage == ATR_STORAGE_F16) launch_wbp_bp_t<_Float16>(p, a, ny, s);
    else if (p.storage == ATR_STORAGE_BF16) launch_wbp_bp_t<bf16_t>(p, a, ny, s);
    else launch_wbp_bp_t<float>(p, a, ny, s);
}

std::vector<BpLaunch> lay_out_bp(const std::vector<QueueEntry<BpItem>>& ent, BpItem* out)
{
    std::vector<BpLaunch> launches;
    int first = 0;
    for (int shape = 0; shape < BP_SHAPES; shape++) {
        std::vector<QueueEntry<BpItem>> g;
        for (const auto& e : ent)
            if (e.item.shape == shape) g.push_back(e);
        if (g.empty()) continue;
        const int total = lay_out_entries(g, out + first);
        launches.push_back(BpLaunch{first, (int)g.size(), total, shape});
        first += (int)g.size();
    }
    return launches;
}

// items == nullptr: resident blocks per CU, else the launch
template <typename S, int SHAPE>
static int bp_batch_v(const BpLaunch* l, const BpItem* items, int* counter, int grid,
                      hipStream_t s)
{
    if (!items) {
        int nb = 0;
        const hipError_t e =
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_back_proj_batch<S, SHAPE>, BP_THREADS, 0);
        return (e == hipSuccess && nb > 0) ? nb : 1;
    }
    hipLaunchKernelGGL((k_back_proj_batch<S, SHAPE>), dim3(grid), dim3(BP_THREADS), 0, s, items,
                       l->n_entries, l->total, counter);
    return 0;
}

template <typename S>
static int bp_batch_s(const BpLaunch* l, const BpItem* items, int* counter, int grid,
                      hipStream_t s)
{
    switch (l->shape) {
    case 1: return bp_batch_v<S, 1>(l, items, counter, grid, s);
    case 2: return bp_batch_v<S, 2>(l, items, counter, grid, s);
    case 3: return bp_batch_v<S, 3>(l, items, counter, grid, s);
    default: return bp_batch_v<S, 0>(l, items, counter, grid, s);
    }
}

static int bp_batch(int storage, const BpLaunch* l, const BpItem* items, int* counter, int grid,
                    hipStream_t s)
{
    if (storage == ATR_STORAGE_F16) return bp_batch_s<_Float16>(l, items, counter, grid, s);
    if (storage == ATR_STORAGE_BF16) return bp_batch_s<bf16_t>(l, items, counter, grid, s);
    return bp_batch_s<float>(l, items, counter, grid, s);
}

void launch_bp_batch(int storage, const BpLaunch& l, const BpItem* items, int* counter, int grid,
                     hipStream_t s)
{
    (void)bp_batch(storage, &l, items, counter, std::max(1, std::min(grid, l.total)), s);
}

int bp_batch_grid(int storage, const BpLaunch& l)
{
    int dev = 0, cus = 1;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        cus = 1;
    return cus * bp_batch(storage, &l, nullptr, nullptr, 0, nullptr);
}

void launch_zero(float* ptr, size_t n, hipStream_t s)
{
    size_t blocks = std::min<size_t>((n + 255) / 256, 65536);
    if (blocks == 0) return;
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)blocks), dim3(256), 0, s, ptr, n);
}

void launch_zero_int(int* ptr, int n, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill_zero_int, dim3((n + 255) / 256), dim3(256), 0, s, ptr, n);
}

void launch_load_volume(const Plan& p, const float* in, hipStream_t s)
{
    size_t n = (size_t)p.vol_x * p.vol_z;
    unsigned bx = (unsigned)std::min<size_t>((n + 255) / 256, 64);
    hipLaunchKernelGGL(k_load_volume, dim3(bx, p.vol_y), dim3(256), 0, s, in, p.d_vol, p.vol_x,
                       p.vol_z, p.d_vflag);
}

void launch_vol_stats(const Plan& p, hipStream_t s)
{
    hipLaunchKernelGGL(k_vol_stats, dim3(p.vol_y), dim3(256), 0, s, p.d_vol, p.vol_x, p.vol_z,
                       p.d_vflag, (double2*)p.d_vstats);
}

void launch_output(const Plan& p, float* out, hipStream_t s)
{
    dim3 grid((p.vol_x + 255) / 256, p.vol_z, p.vol_y);
    hipLaunchKernelGGL(k_output, grid, dim3(256), 0, s, p.d_vol, p.vol_x, p.vol_y, p.vol_z,
                       p.d_vflag, (const double2*)p.d_vstats, p.d_fill_vol, p.layout, out);
}

}  // namespace atr
