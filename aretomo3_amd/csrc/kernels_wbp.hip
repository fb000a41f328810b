// kernels_wbp.hip -- weighted back-projection path (gfx950):
//   k_filter        weighting + ramp/Hamming filter, row FFT
//                   (Recon/GWeightProjs.cu:7-19, Recon/GRWeight.cu:7-69)
//   k_wbp_rowfft    row FFT of two rows of the 2x grid (the back-projection
//                   onto that grid is k_wbp_grid_bp in kernels_sart.hip)
//                   (Recon/GBackProjWbp.cu:126)
//   k_colfft        column FFT, normalisation, crop, inverse column FFT
//                   (MaUtil/CCufft2D.cpp:65-80, MaUtil/GFourierResize2D.cu:7-39)
//   k_wbp_rowc2r    real inverse row FFT + output layout
//                   (MaUtil/CCufft2D.cpp:108-123, MaUtil/CPad2D.cpp:29-39,
//                    Recon/CDoWbpRecon.cpp:107-123)
//   k_bin_*         the same three for the Fourier binning of the aligned stack
// Each has two forms: _reg<N> for powers of two, the transform in registers
// (fft_reg.h), and one over LDS for any other length; both give the same bits.
// Scratch: d_wbp_grid [slab][2VolZ][2VolX]; spectra in blocks of kb columns,
// d_wbp_t [slab][blocks][2VolZ][kb], d_wbp_u [slab][blocks][VolZ][kb], so that a
// column transform's workgroup reads and writes one contiguous range (with
// rows of VolX/2+1 values it read 64-byte pieces across 128-byte lines).
//
// Measured per launch, form over LDS (with integer divisions by the run-time
// lengths) / in registers, MI355X, whose copies reach 4.9 TB/s:
//   filter    61 x 2048 x 2048, FP16          2.14 / 0.63 ms
//   row FFT   36 slices, grid 4096 x 1024     0.83 / 0.27 ms  (3.4 TB/s)
//             512 slices, grid 1024 x 256     0.39 / 0.17 ms  (4.6 TB/s)
//   columns   36 slices 1025 x 1024 -> 512    0.50 / 0.12 ms  (3.8 TB/s)
//             512 slices 257 x 256 -> 128     0.33 / 0.10 ms
//   c2r       36 slices 2048 x 512            0.19 / 0.09 ms
//             512 slices 512 x 128            0.18 / 0.06 ms
//   binning   41 x 4096 x 4096 by 4, rows     5.3 / 1.5 ms, columns 1.6 / 0.31 ms
// All are bound by memory now, the row transforms of long rows in part by the
// two waits for the other waves in each exchange.
#include <algorithm>

#include "atr_internal.h"
#include "fft_reg.h"
#include "storage.h"

namespace atr {

// Value of pixel i, v as read: an empty one takes the first that is not empty
// along the table's chain.
__device__ __forceinline__ float filled_from_w(float v, const float* __restrict__ img, int i,
                                               const int* __restrict__ table, float mean)
{
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
__device__ __forceinline__ float filled_value_w(const float* __restrict__ img, int i,
                                                const int* __restrict__ table, float mean)
{
    return filled_from_w(img[i], img, i, table, mean);
}

// Half spectra in blocks of kb columns, [slice][block][row][kb]: first entry of
// a slice, entry (k, row) of it.
__host__ __device__ __forceinline__ size_t spec_slice(int slice, int columns, int rows, int kb)
{
    return (size_t)slice * ((columns + kb - 1) / kb) * rows * kb;
}
__device__ __forceinline__ size_t spec_at(int k, int row, int rows, int kb)
{
    // kb is a power of two
    const int sh = __builtin_ctz(kb);
    return ((size_t)(k >> sh) * rows + row) * kb + (k & (kb - 1));
}

// Bin k of the spectra of the two real rows that were transformed as one
// complex row, from its points k and N - k: A = (Z[k] + conj Z[N-k]) / 2, B =
// (Z[k] - conj Z[N-k]) / (2i), B one row (kb entries) further.
__device__ __forceinline__ void spec_split(float2* dst, int kb, float2 z1, float2 z2, bool both)
{
    dst[0] = make_float2(0.5f * (z1.x + z2.x), 0.5f * (z1.y - z2.y));
    if (both) dst[kb] = make_float2(0.5f * (z1.y + z2.y), -0.5f * (z1.x - z2.x));
}

// Point k of the complex row A + iB whose real inverse transforms are rows
// `row` and `row` + 1 of n points (imaginary parts of the DC and Nyquist bins
// are ignored, numpy irfft).
__device__ __forceinline__ float2 spec_join(const float2* h, int k, int n, int row, int rows, int kb,
                                            bool both)
{
    const int half = n / 2, m = k <= half ? k : n - k;
    const float2* p = h + spec_at(m, row, rows, kb);
    float2 a = p[0], b = both ? p[kb] : make_float2(0.0f, 0.0f);
    if (m == 0 || m == half) a.y = b.y = 0.0f;
    else if (k > half) a.y = -a.y, b.y = -b.y;
    return make_float2(a.x - b.y, a.y + b.x);
}

// ------------------------------------------------------------------------
// Fourier binning of the aligned stack (Correct/CBinStack.cpp:54-106,
// -AtBin > 1): per image, R2C over ax x ay normalised by 1/(ax ay), crop to
// bx x by (MaUtil/GFourierResize2D.cu:7-39), unnormalised C2R.
//   k_bin_rowfft  two image rows packed as one complex row, FFT of length
//                 ax, the columns kx < bx/2+1 of both half spectra kept
//   k_colfft      per block of columns: FFT of length ay, normalisation,
//                 crop to by rows, inverse FFT of length by
//   k_bin_rowc2r  two binned rows: packed C2R of length bx
// ------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_bin_rowfft(const float* __restrict__ in, size_t tilt_stride,
                                                    size_t row_stride, int fill,
                                                    const int* __restrict__ table,
                                                    const double2* __restrict__ tilt_stats,
                                                    int ax, int ay, int kxb, int kb, FftDesc fd,
                                                    float2* __restrict__ tbuf)
{
    extern __shared__ float2 lds[];
    float2* a = lds;
    float2* b = lds + ax;
    const int t = blockIdx.y;
    const int y0 = 2 * blockIdx.x, y1 = y0 + 1;
    const bool has1 = y1 < ay;
    const float* img = in + (size_t)t * tilt_stride;
    float mean = 0.0f;
    if (fill) {
        double2 ts = tilt_stats[t];
        mean = ts.y > 0 ? (float)(ts.x / ts.y) : 0.0f;
    }
    for (int x = threadIdx.x; x < ax; x += blockDim.x) {
        float va, vb = 0.0f;
        if (fill) {
            va = filled_value_w(img, (int)(y0 * row_stride + x), table, mean);
            if (has1) vb = filled_value_w(img, (int)(y1 * row_stride + x), table, mean);
        } else {
            va = img[(size_t)y0 * row_stride + x];
            if (has1) vb = img[(size_t)y1 * row_stride + x];
        }
        a[x] = make_float2(va, vb);
    }
    __syncthreads();
    float2* r = lds_fft(a, b, fd, 1, -1.0f, threadIdx.x, blockDim.x);
    float2* dst = tbuf + spec_slice(t, kxb, ay, kb);
    for (int k = threadIdx.x; k < kxb; k += blockDim.x)
        spec_split(dst + spec_at(k, y0, ay, kb), kb, r[k], r[k ? ax - k : 0], has1);
}

// Column transforms, n rows cropped to m (row j <= m/2 from j, else from j - m
// + n), for a block of kb columns: forward, times norm, inverse.  The binning
// (n = ay, m = by) and the WBP (n = 2 VolZ, m = VolZ).
__global__ __launch_bounds__(256) void k_colfft(const float2* __restrict__ tbuf,
                                                float2* __restrict__ ubuf, int n, int m, int kb,
                                                float norm, FftDesc fn, FftDesc fm)
{
    extern __shared__ float2 lds[];
    float2* a = lds;
    float2* b = lds + kb * n;
    const size_t blk = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    const float2* src = tbuf + blk * n * kb;
    const float inv_kb = 1.0f / (float)kb, inv_m = 1.0f / (float)m;
    for (int i = threadIdx.x; i < kb * n; i += blockDim.x) {
        const int z = fft_div(i, inv_kb), col = i - z * kb;
        a[col * n + z] = src[i];
    }
    __syncthreads();
    float2* r = lds_fft(a, b, fn, kb, -1.0f, threadIdx.x, blockDim.x);
    float2* o = (r == a) ? b : a;
    for (int i = threadIdx.x; i < kb * m; i += blockDim.x) {
        const int col = fft_div(i, inv_m), j = i - col * m;
        const float2 v = r[col * n + (j <= m / 2 ? j : j - m + n)];
        o[col * m + j] = make_float2(v.x * norm, v.y * norm);
    }
    __syncthreads();
    float2* q = lds_fft(o, r, fm, kb, 1.0f, threadIdx.x, blockDim.x);
    float2* dst = ubuf + blk * m * kb;
    for (int i = threadIdx.x; i < kb * m; i += blockDim.x) {
        const int z = fft_div(i, inv_kb), col = i - z * kb;
        dst[i] = q[col * m + z];
    }
}

// The same in registers: thread = (column, t), entry i of a column's LDS at
// fft_pad(i) KB + column.  M: the inverse's length, whose transforms take the
// first KB M / 16 threads.
template <int N, int M, int KB>
__global__ __launch_bounds__(KB * (N / 16)) void k_colfft_reg(const float2* __restrict__ tbuf,
                                                              float2* __restrict__ ubuf, float norm,
                                                              const float2* __restrict__ tw_n,
                                                              const float2* __restrict__ tw_m)
{
    constexpr int T = N / 16, TM = M / 16;
    extern __shared__ float2 lds[];
    const int col = threadIdx.x % KB, t = threadIdx.x / KB;
    const size_t blk = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    const float2* src = tbuf + blk * N * KB + col;
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = src[(t + q * T) * KB];
    fft_run<N, KB, false>(v, t, tw_n, -1.0f, lds + col);
    __syncthreads();
    // crop: rows up to M/2 stay, rows above N - M/2 move down by N - M
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int i = t + q * T;
        const int j = i <= M / 2 ? i : i - N + M;
        if (j > M / 2 || i <= M / 2)
            lds[fft_pad(j) * KB + col] = make_float2(v[q].x * norm, v[q].y * norm);
    }
    __syncthreads();
    const bool active = t < TM;
    if (active) {
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = lds[fft_pad(t + q * TM) * KB + col];
    }
    fft_run<M, KB, false>(v, t, tw_m, 1.0f, lds + col, active);
    if (active) {
        float2* dst = ubuf + blk * M * KB + col;
#pragma unroll
        for (int q = 0; q < 16; q++) dst[(t + q * TM) * KB] = v[q];
    }
}

__global__ __launch_bounds__(256) void k_bin_rowc2r(const float2* __restrict__ ubuf, int bx, int by,
                                                    int kb, FftDesc fx, float* __restrict__ out)
{
    extern __shared__ float2 lds[];
    float2* a = lds;
    float2* b = lds + bx;
    const int t = blockIdx.y, ya = 2 * blockIdx.x, yb = ya + 1;
    const bool has_b = yb < by;
    const float2* h = ubuf + spec_slice(t, bx / 2 + 1, by, kb);
    for (int k = threadIdx.x; k < bx; k += blockDim.x)
        a[k] = spec_join(h, k, bx, ya, by, kb, has_b);
    __syncthreads();
    float2* r = lds_fft(a, b, fx, 1, 1.0f, threadIdx.x, blockDim.x);
    float* oa = out + ((size_t)t * by + ya) * bx;
    for (int x = threadIdx.x; x < bx; x += blockDim.x) {
        oa[x] = r[x].x;
        if (has_b) oa[bx + x] = r[x].y;
    }
}

// Points t + q N/16 of two rows of an image as one complex row.  All values are
// loaded before the first is looked at for the fill of empty pixels (a load at a
// time in flight otherwise).
template <int N>
__device__ __forceinline__ void load_row_pair(float2 (&v)[16], const float* __restrict__ img,
                                              size_t row_stride, int y0, bool has1, int t, int fill,
                                              const int* __restrict__ table, float mean)
{
    constexpr int T = N / 16;
    const size_t r0 = y0 * row_stride, r1 = r0 + (has1 ? row_stride : 0);
#pragma unroll
    for (int q = 0; q < 16; q++)
        v[q] = make_float2(img[r0 + t + q * T], has1 ? img[r1 + t + q * T] : 0.0f);
    if (!fill) return;
    float low = v[0].x;
#pragma unroll
    for (int q = 0; q < 16; q++) low = fminf(low, fminf(v[q].x, v[q].y));
    if (!(low < kEmpty)) return;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        v[q].x = filled_from_w(v[q].x, img, (int)r0 + t + q * T, table, mean);
        if (has1) v[q].y = filled_from_w(v[q].y, img, (int)r1 + t + q * T, table, mean);
    }
}

template <int N>
__global__ __launch_bounds__(fft_row_threads(N)) void k_bin_rowfft_reg(
    const float* __restrict__ in, size_t tilt_stride, size_t row_stride, int fill,
    const int* __restrict__ table, const double2* __restrict__ tilt_stats, int ay, int kxb, int kb,
    const float2* __restrict__ tw, float2* __restrict__ tbuf)
{
    constexpr int T = N / 16, F = fft_rows(N);
    constexpr bool WAVE = fft_in_wave(N);
    extern __shared__ float2 lds[];
    const int f = threadIdx.x / T, t = threadIdx.x % T, tilt = blockIdx.y;
    const int y0 = min(2 * (int)(blockIdx.x * F + f), ay - 1);
    const bool has = 2 * (int)(blockIdx.x * F + f) < ay, has1 = y0 + 1 < ay;
    float2* buf = lds + f * fft_reg_lds(N);
    const float* img = in + (size_t)tilt * tilt_stride;
    float mean = 0.0f;
    if (fill) {
        const double2 ts = tilt_stats[tilt];
        mean = ts.y > 0 ? (float)(ts.x / ts.y) : 0.0f;
    }
    float2 v[16];
    load_row_pair<N>(v, img, row_stride, y0, has1, t, fill, table, mean);
    fft_run<N, 1, WAVE>(v, t, tw, -1.0f, buf);
    fft_sync<WAVE>();
#pragma unroll
    for (int q = 0; q < 16; q++) buf[fft_pad(t + q * T)] = v[q];
    fft_sync<WAVE>();
    if (!has) return;
    float2* dst = tbuf + spec_slice(tilt, kxb, ay, kb);
    for (int k = t; k < kxb; k += T)
        spec_split(dst + spec_at(k, y0, ay, kb), kb, buf[fft_pad(k)], buf[fft_pad(k ? N - k : 0)],
                   has1);
}

template <int N>
__global__ __launch_bounds__(fft_row_threads(N)) void k_bin_rowc2r_reg(const float2* __restrict__ ubuf,
                                                                       int by, int kb,
                                                                       const float2* __restrict__ tw,
                                                                       float* __restrict__ out)
{
    constexpr int T = N / 16, F = fft_rows(N);
    constexpr bool WAVE = fft_in_wave(N);
    extern __shared__ float2 lds[];
    const int f = threadIdx.x / T, t = threadIdx.x % T, tilt = blockIdx.y;
    const int ya = min(2 * (int)(blockIdx.x * F + f), by - 1);
    const bool has = 2 * (int)(blockIdx.x * F + f) < by, has_b = ya + 1 < by;
    const float2* h = ubuf + spec_slice(tilt, N / 2 + 1, by, kb);
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = spec_join(h, t + q * T, N, ya, by, kb, has_b);
    fft_run<N, 1, WAVE>(v, t, tw, 1.0f, lds + f * fft_reg_lds(N));
    if (!has) return;
    float* oa = out + ((size_t)tilt * by + ya) * N;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        oa[t + q * T] = v[q].x;
        if (has_b) oa[N + t + q * T] = v[q].y;
    }
}

// A product that is not fused into the sum that takes it (in the form over LDS
// it is stored in between).
__device__ __forceinline__ float rounded(float x)
{
    asm("" : "+v"(x));
    return x;
}

// k_filter in registers: the forward transform leaves each thread the points
// that the inverse starts from.
template <typename S, int N>
__global__ __launch_bounds__(fft_row_threads(N)) void k_filter_reg(
    const float* __restrict__ in, size_t tilt_stride, size_t row_stride, int fill,
    const int* __restrict__ table, const double2* __restrict__ tilt_stats,
    const float2* __restrict__ cs, int n, int rows, int vol_z, const float2* __restrict__ tw,
    const float* __restrict__ filt, S* __restrict__ sino, int stride, int* __restrict__ sflag)
{
    constexpr int T = N / 16, F = fft_rows(N);
    constexpr bool WAVE = fft_in_wave(N);
    extern __shared__ float2 lds[];
    const int f = threadIdx.x / T, t = threadIdx.x % T, tilt = blockIdx.y;
    const int y0 = min(2 * (int)(blockIdx.x * F + f), rows - 1);
    const bool has = 2 * (int)(blockIdx.x * F + f) < rows, has1 = y0 + 1 < rows;
    float2* buf = lds + f * fft_reg_lds(N);
    const float w = cs[tilt].x / (float)vol_z;
    const float* img = in + (size_t)tilt * tilt_stride;
    float mean = 0.0f;
    if (fill) {
        const double2 ts = tilt_stats[tilt];
        mean = ts.y > 0 ? (float)(ts.x / ts.y) : 0.0f;
    }
    float2 v[16];
    load_row_pair<N>(v, img, row_stride, y0, has1, t, fill, table, mean);
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = make_float2(rounded(v[q].x * w), rounded(v[q].y * w));
    fft_run<N, 1, WAVE>(v, t, tw, -1.0f, buf);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int k = t + q * T;
        const float g = filt[k <= N / 2 ? k : N - k];
        v[q] = make_float2(rounded(v[q].x * g), rounded(v[q].y * g));
    }
    fft_run<N, 1, WAVE>(v, t, tw, 1.0f, buf);
    if (!has) return;
    S* d0 = sino + ((size_t)y0 * n + tilt) * stride;
    S* d1 = sino + ((size_t)(y0 + 1) * n + tilt) * stride;
    bool sent = false;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        sent |= v[q].x <= kEmpty;
        st<S>(d0 + t + q * T, v[q].x);
        if (has1) {
            sent |= v[q].y <= kEmpty;
            st<S>(d1 + t + q * T, v[q].y);
        }
    }
    if (sent) {
        atomicOr(sflag + y0, 1);
        if (has1) atomicOr(sflag + y0 + 1, 1);
    }
    // (N is a multiple of 64, the row stride: no padding to clear)
}

// One workgroup per (tilt, pair of rows): the two weighted rows are packed as
// real and imaginary parts of one complex row, transformed, scaled by the
// real even filter (which keeps the two parts separate), transformed back.
template <typename S>
__global__ __launch_bounds__(256) void k_filter(const float* __restrict__ in, size_t tilt_stride,
                                                size_t row_stride, int fill,
                                                const int* __restrict__ table,
                                                const double2* __restrict__ tilt_stats,
                                                const float2* __restrict__ cs, int n, int rows,
                                                int proj, int vol_z, FftDesc fd,
                                                const float* __restrict__ filt,
                                                S* __restrict__ sino, int stride,
                                                int* __restrict__ sflag)
{
    extern __shared__ float2 lds[];
    float2* a = lds;
    float2* b = lds + proj;
    const int t = blockIdx.y;
    const int y0 = 2 * blockIdx.x, y1 = y0 + 1;
    const bool has1 = y1 < rows;
    const float w = cs[t].x / (float)vol_z;
    const float* img = in + (size_t)t * tilt_stride;
    float mean = 0.0f;
    if (fill) {
        double2 ts = tilt_stats[t];
        mean = ts.y > 0 ? (float)(ts.x / ts.y) : 0.0f;
    }
    for (int x = threadIdx.x; x < proj; x += blockDim.x) {
        float va, vb = 0.0f;
        if (fill) {
            va = filled_value_w(img, (int)(y0 * row_stride + x), table, mean);
            if (has1) vb = filled_value_w(img, (int)(y1 * row_stride + x), table, mean);
        } else {
            va = img[(size_t)y0 * row_stride + x];
            if (has1) vb = img[(size_t)y1 * row_stride + x];
        }
        a[x] = make_float2(va * w, vb * w);
    }
    __syncthreads();
    float2* r = lds_fft(a, b, fd, 1, -1.0f, threadIdx.x, blockDim.x);
    for (int k = threadIdx.x; k < proj; k += blockDim.x) {
        int kk = k <= proj / 2 ? k : proj - k;
        float f = filt[kk];
        r[k] = make_float2(r[k].x * f, r[k].y * f);
    }
    __syncthreads();
    float2* o = (r == a) ? b : a;
    r = lds_fft(r, o, fd, 1, 1.0f, threadIdx.x, blockDim.x);
    S* d0 = sino + ((size_t)y0 * n + t) * stride;
    S* d1 = sino + ((size_t)y1 * n + t) * stride;
    bool sent = false;
    for (int x = threadIdx.x; x < stride; x += blockDim.x) {
        float va = x < proj ? r[x].x : 0.0f;
        float vb = x < proj ? r[x].y : 0.0f;
        sent |= va <= kEmpty;
        st<S>(d0 + x, va);
        if (has1) {
            sent |= vb <= kEmpty;
            st<S>(d1 + x, vb);
        }
    }
    if (sent) {
        atomicOr(sflag + y0, 1);
        if (has1) atomicOr(sflag + y1, 1);
    }
}

// One workgroup per (slice, pair of 2x-grid rows).  Every grid point is the
// mean of the linear interpolations of the tilts whose FP64 inclusion
// interval holds it (0 when none).  The two rows are transformed together as
// one complex row of length 2VolX; bins 0..VolX/2 of each are written.
// Row FFT of the 2x grid (Recon/GBackProjWbp.cu:126-130 forward R2C along x):
// two grid rows packed as one complex row, one LDS FFT of length 2 VolX, the
// two half spectra split apart.
__global__ __launch_bounds__(256) void k_wbp_rowfft(const float* __restrict__ grid, int vol_x,
                                                    int vol_z, int kb, FftDesc fd,
                                                    float2* __restrict__ tbuf)
{
    extern __shared__ float2 lds[];
    const int nx2 = 2 * vol_x, nz2 = 2 * vol_z, kxn = vol_x / 2 + 1;
    float2* a = lds;
    float2* b = lds + nx2;
    const int zp = blockIdx.x, ys = blockIdx.y;
    const int za = 2 * zp;
    const float* ra = grid + ((size_t)ys * nz2 + za) * nx2;
    const float* rb = ra + nx2;
    for (int x = threadIdx.x; x < nx2; x += blockDim.x) a[x] = make_float2(ra[x], rb[x]);
    __syncthreads();
    float2* r = lds_fft(a, b, fd, 1, -1.0f, threadIdx.x, blockDim.x);
    float2* dst = tbuf + spec_slice(ys, kxn, nz2, kb);
    for (int k = threadIdx.x; k < kxn; k += blockDim.x)
        spec_split(dst + spec_at(k, za, nz2, kb), kb, r[k], r[k ? nx2 - k : 0], true);
}

// Row FFT of the 2x grid in registers, N = 2 VolX; fft_rows(N) row pairs per
// workgroup.  Only bins 0 .. VolX/2 of each half spectrum are kept: point k and
// its mirror N - k, so a thread exchanges the last quarter of its points only.
template <int N>
__global__ __launch_bounds__(fft_row_threads(N)) void k_wbp_rowfft_reg(
    const float* __restrict__ grid, int vol_z, int kb, const float2* __restrict__ tw,
    float2* __restrict__ tbuf)
{
    constexpr int T = N / 16, F = fft_rows(N);
    constexpr bool WAVE = fft_in_wave(N);
    __shared__ float2 lds[F * fft_reg_lds(N)];
    const int f = threadIdx.x / T, t = threadIdx.x % T, ys = blockIdx.y;
    const int zp = blockIdx.x * F + f, nz2 = 2 * vol_z, kxn = N / 4 + 1;
    const bool has = zp < vol_z;
    const int za = 2 * min(zp, vol_z - 1);
    float2* buf = lds + f * fft_reg_lds(N);
    const float* ra = grid + ((size_t)ys * nz2 + za) * N;
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = make_float2(ra[t + q * T], ra[N + t + q * T]);
    fft_run<N, 1, WAVE>(v, t, tw, -1.0f, buf);
    fft_sync<WAVE>();
#pragma unroll
    for (int q = 12; q < 16; q++) buf[fft_pad(t + q * T)] = v[q];
    fft_sync<WAVE>();
    if (!has) return;
    float2* dst = tbuf + spec_slice(ys, kxn, nz2, kb);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int k = t + q * T;
        spec_split(dst + spec_at(k, za, nz2, kb), kb, v[q], k ? buf[fft_pad(N - k)] : v[0], true);
    }
    if (t == 0)
        spec_split(dst + spec_at(N / 4, za, nz2, kb), kb, v[4], buf[fft_pad(3 * (N / 4))], true);
}

__device__ __forceinline__ size_t out_index_w(int layout, int x, int y, int z, int vol_x,
                                              int vol_y, int vol_z)
{
    switch (layout) {
    case ATR_LAYOUT_XYZ: return ((size_t)z * vol_y + y) * vol_x + x;
    case ATR_LAYOUT_XYZ_NOFLIP: return ((size_t)(vol_z - 1 - z) * vol_y + y) * vol_x + x;
    case ATR_LAYOUT_SLICE: return ((size_t)y * vol_z + z) * vol_x + x;
    default: return ((size_t)y * vol_z + (vol_z - 1 - z)) * vol_x + x;
    }
}

// One workgroup per (slice, pair of output rows): the unnormalised C2R of
// length VolX of two half spectra, packed as one complex inverse FFT.  The
// imaginary parts of the DC and Nyquist bins are ignored (numpy irfft).
__global__ __launch_bounds__(256) void k_wbp_rowc2r(const float2* __restrict__ ubuf, int vol_x,
                                                    int vol_y, int vol_z, int y0, int kb, FftDesc fx,
                                                    int layout, float* __restrict__ out)
{
    extern __shared__ float2 lds[];
    float2* a = lds;
    float2* b = lds + vol_x;
    const int zp = blockIdx.x, ys = blockIdx.y, y = y0 + ys;
    const int za = 2 * zp, zb = za + 1;
    const bool has_b = zb < vol_z;
    const float2* h = ubuf + spec_slice(ys, vol_x / 2 + 1, vol_z, kb);
    for (int k = threadIdx.x; k < vol_x; k += blockDim.x)
        a[k] = spec_join(h, k, vol_x, za, vol_z, kb, has_b);
    __syncthreads();
    float2* r = lds_fft(a, b, fx, 1, 1.0f, threadIdx.x, blockDim.x);
    for (int x = threadIdx.x; x < vol_x; x += blockDim.x) {
        out[out_index_w(layout, x, y, za, vol_x, vol_y, vol_z)] = r[x].x;
        if (has_b) out[out_index_w(layout, x, y, zb, vol_x, vol_y, vol_z)] = r[x].y;
    }
}

template <int N>
__global__ __launch_bounds__(fft_row_threads(N)) void k_wbp_rowc2r_reg(
    const float2* __restrict__ ubuf, int vol_y, int vol_z, int y0, int kb,
    const float2* __restrict__ tw, int layout, float* __restrict__ out)
{
    constexpr int T = N / 16, F = fft_rows(N);
    constexpr bool WAVE = fft_in_wave(N);
    extern __shared__ float2 lds[];
    const int f = threadIdx.x / T, t = threadIdx.x % T, ys = blockIdx.y, y = y0 + ys;
    const int za = min(2 * (int)(blockIdx.x * F + f), vol_z - 1);
    const bool has = 2 * (int)(blockIdx.x * F + f) < vol_z, has_b = za + 1 < vol_z;
    const float2* h = ubuf + spec_slice(ys, N / 2 + 1, vol_z, kb);
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = spec_join(h, t + q * T, N, za, vol_z, kb, has_b);
    fft_run<N, 1, WAVE>(v, t, tw, 1.0f, lds + f * fft_reg_lds(N));
    if (!has) return;
    float* oa = out + out_index_w(layout, 0, y, za, N, vol_y, vol_z);
    float* ob = out + out_index_w(layout, 0, y, has_b ? za + 1 : za, N, vol_y, vol_z);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        oa[t + q * T] = v[q].x;
        if (has_b) ob[t + q * T] = v[q].y;
    }
}

// ------------------------------------------------------------------------
// fn(std::integral_constant<int, N>) for the power of two n of [64, 8192]; false
// for any other n, whose transforms go over LDS (2 to 4 times the time per point,
// but any prime factor).
template <int N = 64, class F>
static bool with_pow2(int n, F&& fn)
{
    if constexpr (N <= 8192) {
        if (n == N) {
            fn(std::integral_constant<int, N>{});
            return true;
        }
        return with_pow2<2 * N>(n, fn);
    }
    return false;
}

// Grid of row transforms over `pairs` row pairs and LDS of a workgroup.
template <int N>
static dim3 row_grid(int pairs, int batch)
{
    return dim3((pairs + fft_rows(N) - 1) / fft_rows(N), batch);
}
template <int N>
static constexpr size_t row_lds() { return (size_t)fft_rows(N) * fft_reg_lds(N) * sizeof(float2); }

template <int N, int M, int KB>
static void launch_col_reg(const float2* tbuf, float2* ubuf, int blocks, int batch, float norm,
                           const float2* tw_n, const float2* tw_m, hipStream_t s)
{
    const size_t shm = (size_t)KB * fft_reg_lds(N) * sizeof(float2);
    hipLaunchKernelGGL((k_colfft_reg<N, M, KB>), dim3(blocks, batch), dim3(KB * (N / 16)), shm, s,
                       tbuf, ubuf, norm, tw_n, tw_m);
}

// Column transforms of `batch` slices, n rows to m: in registers where both are
// powers of two and m is a half (all WBP crops), a quarter or an eighth of n --
// another crop would leave more than 7/8 of the inverse's threads idle or need
// its own instances -- and over LDS otherwise.
static void launch_cols(const float2* tbuf, float2* ubuf, int columns, int batch, int n, int m, int kb,
                        float norm, const FftDesc& fn, const FftDesc& fm, hipStream_t s)
{
    const int blocks = (columns + kb - 1) / kb;
    if (fft_col_reg_ok(n, m)) {
        with_pow2(n, [&](auto nc) {
            constexpr int N = decltype(nc)::value;
            with_pow2(m, [&](auto mc) {
                constexpr int M = decltype(mc)::value;
                if constexpr (fft_col_reg_ok(N, M))
                    launch_col_reg<N, M, fft_col_reg_width(N)>(tbuf, ubuf, blocks, batch, norm, fn.tw,
                                                               fm.tw, s);
            });
        });
        return;
    }
    const size_t shm = 2 * (size_t)kb * n * sizeof(float2);
    hipLaunchKernelGGL(k_colfft, dim3(blocks, batch), dim3(256), shm, s, tbuf, ubuf, n, m, kb, norm, fn,
                       fm);
}

template <typename S>
static void launch_filter_t(const Plan& p, const float* in, hipStream_t s)
{
    const StageSource src0 = stage_source(p, in);
    const float* src = src0.src;
    const size_t ts = src0.tilt_stride, rs = src0.row_stride;
    if (with_pow2(p.proj, [&](auto nc) {
            constexpr int N = decltype(nc)::value;
            if constexpr (N <= WBP_MAX)
                hipLaunchKernelGGL((k_filter_reg<S, N>), row_grid<N>((p.vol_y + 1) / 2, p.n),
                                   dim3(fft_row_threads(N)), row_lds<N>(), s, src, ts, rs,
                                   src0.fill ? 1 : 0, p.d_fill_aln, (const double2*)p.d_tilt_stats,
                                   p.d_cs, p.n, p.vol_y, p.vol_z, p.d_tw_proj, p.d_filter,
                                   (S*)p.d_sino, p.sino_stride, p.d_sflag);
        }))
        return;
    dim3 grid((p.vol_y + 1) / 2, p.n);
    size_t shm = 2 * (size_t)p.proj * sizeof(float2);
    hipLaunchKernelGGL(k_filter<S>, grid, dim3(256), shm, s, src, ts, rs, src0.fill ? 1 : 0,
                       p.d_fill_aln, (const double2*)p.d_tilt_stats, p.d_cs, p.n, p.vol_y, p.proj,
                       p.vol_z, p.fft_proj, p.d_filter, (S*)p.d_sino, p.sino_stride, p.d_sflag);
}

void launch_filter_wbp(const Plan& p, const float* in, hipStream_t s)
{
    if (p.storage == ATR_STORAGE_F16) launch_filter_t<_Float16>(p, in, s);
    else if (p.storage == ATR_STORAGE_BF16) launch_filter_t<bf16_t>(p, in, s);
    else launch_filter_t<float>(p, in, s);
}

void launch_wbp_rowfft(const Plan& p, int ny, hipStream_t s)
{
    if (with_pow2(2 * p.vol_x, [&](auto nc) {
            constexpr int N = decltype(nc)::value;
            if constexpr (N <= 2 * WBP_MAX)
                hipLaunchKernelGGL(k_wbp_rowfft_reg<N>, row_grid<N>(p.vol_z, ny),
                                   dim3(fft_row_threads(N)), 0, s, p.d_wbp_grid, p.vol_z, p.wbp_kb,
                                   p.d_tw_x2, p.d_wbp_t);
        }))
        return;
    dim3 grid(p.vol_z, ny);
    size_t shm = 2 * (size_t)(2 * p.vol_x) * sizeof(float2);
    hipLaunchKernelGGL(k_wbp_rowfft, grid, dim3(256), shm, s, p.d_wbp_grid, p.vol_x, p.vol_z, p.wbp_kb,
                       p.fft_x2, p.d_wbp_t);
}

void launch_wbp_colfft(const Plan& p, int y0, int ny, hipStream_t s)
{
    (void)y0;
    const float norm = (float)(1.0 / ((double)(2 * p.vol_x) * (double)(2 * p.vol_z)));
    launch_cols(p.d_wbp_t, p.d_wbp_u, p.vol_x / 2 + 1, ny, 2 * p.vol_z, p.vol_z, p.wbp_kb, norm,
                p.fft_z2, p.fft_z, s);
}

void launch_wbp_rowc2r(const Plan& p, int y0, int ny, float* out, hipStream_t s)
{
    if (with_pow2(p.vol_x, [&](auto nc) {
            constexpr int N = decltype(nc)::value;
            if constexpr (N <= WBP_MAX)
                hipLaunchKernelGGL(k_wbp_rowc2r_reg<N>, row_grid<N>((p.vol_z + 1) / 2, ny),
                                   dim3(fft_row_threads(N)), row_lds<N>(), s, p.d_wbp_u, p.vol_y,
                                   p.vol_z, y0, p.wbp_kb, p.d_tw_x, p.layout, out);
        }))
        return;
    dim3 grid((p.vol_z + 1) / 2, ny);
    size_t shm = 2 * (size_t)p.vol_x * sizeof(float2);
    hipLaunchKernelGGL(k_wbp_rowc2r, grid, dim3(256), shm, s, p.d_wbp_u, p.vol_x, p.vol_y,
                       p.vol_z, y0, p.wbp_kb, p.fft_x, p.layout, out);
}

// Fourier binning of the stage input into p.d_binned.
void launch_bin(const Plan& p, const float* in, hipStream_t s)
{
    const float* src = p.prestage ? p.d_aligned : in;
    size_t ts = p.prestage ? (size_t)p.aln_x * p.aln_y : p.in_tilt_stride;
    size_t rs = p.prestage ? (size_t)p.aln_x : p.in_row_stride;
    const int ax = p.aln_x, ay = p.aln_y, bx = p.bin_x, by = p.bin_y, kb = p.bin_kb;
    const int kxb = bx / 2 + 1;
    const double2* stats = (const double2*)p.d_tilt_stats;
    if (!with_pow2(ax, [&](auto nc) {
            constexpr int N = decltype(nc)::value;
            hipLaunchKernelGGL(k_bin_rowfft_reg<N>, row_grid<N>((ay + 1) / 2, p.n),
                               dim3(fft_row_threads(N)), row_lds<N>(), s, src, ts, rs, p.fill ? 1 : 0,
                               p.d_fill_aln, stats, ay, kxb, kb, p.fft_bin_ax.tw, p.d_bin_t);
        })) {
        const size_t shm = 2 * (size_t)ax * sizeof(float2);
        hipLaunchKernelGGL(k_bin_rowfft, dim3((ay + 1) / 2, p.n), dim3(256), shm, s, src, ts, rs,
                           p.fill ? 1 : 0, p.d_fill_aln, stats, ax, ay, kxb, kb, p.fft_bin_ax, p.d_bin_t);
    }
    launch_cols(p.d_bin_t, p.d_bin_u, kxb, p.n, ay, by, kb, (float)(1.0 / ((double)ax * (double)ay)),
                p.fft_bin_ay, p.fft_bin_by, s);
    if (!with_pow2(bx, [&](auto nc) {
            constexpr int N = decltype(nc)::value;
            hipLaunchKernelGGL(k_bin_rowc2r_reg<N>, row_grid<N>((by + 1) / 2, p.n),
                               dim3(fft_row_threads(N)), row_lds<N>(), s, p.d_bin_u, by, kb,
                               p.fft_bin_bx.tw, p.d_binned);
        })) {
        const size_t shm = 2 * (size_t)bx * sizeof(float2);
        hipLaunchKernelGGL(k_bin_rowc2r, dim3((by + 1) / 2, p.n), dim3(256), shm, s, p.d_bin_u, bx, by,
                           kb, p.fft_bin_bx, p.d_binned);
    }
}

size_t spec_elems(int columns, int rows, int kb) { return spec_slice(1, columns, rows, kb); }

}  // namespace atr
