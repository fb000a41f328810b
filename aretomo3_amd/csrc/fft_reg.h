// fft_reg.h -- power-of-two FFTs (64 .. 8192) held in registers (gfx950).
//
// N / 16 threads hold one transform, 16 points each: thread t has the points
// t + q N/16.  A pass is two stages of the LDS transform of fft_lds.h (radix 4
// by 4, and at the end 4 by 2, 4 or 2 as N asks), with that transform's
// butterflies, twiddles and order of operations, so both give the same bits.
// Data go through LDS between passes only: two exchanges for 512 .. 4096
// points instead of a read and a write per radix-4 stage, and the first
// pass takes its points from wherever the caller loads them, the last one
// leaves them in registers.  All indices are shifts and constants; the
// general transform's divisions cost more than its butterflies.
//
// LDS index i lies at i + i / 16: the first pass writes 16 points per thread
// in a row, which would otherwise share two banks.
#pragma once
#include "fft_lds.h"

__device__ __forceinline__ constexpr int fft_pad(int i) { return i + (i >> 4); }
constexpr bool fft_reg_ok(int n) { return n >= 64 && n <= 8192 && (n & (n - 1)) == 0; }
// LDS entries of one transform
constexpr int fft_reg_lds(int n) { return n + n / 16; }

__device__ __forceinline__ float2 fft_tw(const float2* __restrict__ tw, int i, float sign)
{
    float2 w = tw[i];
    w.y *= sign;
    return w;
}

// Radix of the pass that starts with NS finished points: 16 while it fits.
constexpr int fft_pass_radix(int n, int ns) { return n / ns >= 16 ? 16 : n / ns; }

// Position of point q of thread t after the pass (and of the LDS exchange).
template <int N, int NS>
__device__ __forceinline__ int fft_out(int t, int q)
{
    constexpr int R = fft_pass_radix(N, NS);
    if constexpr (R == 16) return (t / NS) * (16 * NS) + (t & (NS - 1)) + q * NS;
    // shorter radices occur in the last pass only, which needs no exchange
    else return t + (N / 16) * q;
}

// One pass on v.  On return v[q] is the point at fft_out<N, NS>(t, q).  After the
// last pass that is t + q N/16, whatever its radix (NS = N / 16 with radix 16).
template <int N, int NS>
__device__ __forceinline__ void fft_pass(float2 (&v)[16], int t, const float2* __restrict__ tw,
                                         float sign)
{
    constexpr int R = fft_pass_radix(N, NS);
    if constexpr (R == 2) {
        // butterflies t + i N/16, i < 8: points i and i + 8
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int k = t + i * (N / 16);
            const float2 a = v[i], b = cmul(v[i + 8], fft_tw(tw, k, sign));
            v[i] = cadd(a, b);
            v[i + 8] = csub(a, b);
        }
    } else {
        // radix 4: butterflies t + i N/16, i < 4: points i, i + 4, i + 8, i + 12
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float2 b[4] = {v[i], v[i + 4], v[i + 8], v[i + 12]};
            if constexpr (NS > 1) {
                const int k = (t + i * (N / 16)) & (NS - 1);
#pragma unroll
                for (int r = 1; r < 4; r++) b[r] = cmul(b[r], fft_tw(tw, r * k * (N / (4 * NS)), sign));
            }
            dft_small<4>(b, sign);
#pragma unroll
            for (int r = 0; r < 4; r++) v[i + 4 * r] = b[r];
        }
        if constexpr (R == 16) {
            // v[i + 4 c]: output c of butterfly i.  The second stage's
            // butterfly c takes output c of the four
            const int k = t & (NS - 1);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                float2 b[4] = {v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]};
                const int kc = k + c * NS;
                if (NS > 1 || c > 0) {
#pragma unroll
                    for (int r = 1; r < 4; r++)
                        b[r] = cmul(b[r], fft_tw(tw, r * kc * (N / (16 * NS)), sign));
                }
                dft_small<4>(b, sign);
#pragma unroll
                for (int r = 0; r < 4; r++) v[4 * c + r] = b[r];
            }
            // output q = c + 4 r
            float2 o[16];
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) o[c + 4 * r] = v[4 * c + r];
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = o[q];
        } else if constexpr (R == 8) {
            // radix 2 on output c of butterflies u and u + N/8 (u = t, t + N/16)
            float2 o[16];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int kc = t + h * (N / 16) + c * NS;
                    const float2 a = v[h + 4 * c], b = cmul(v[h + 2 + 4 * c], fft_tw(tw, kc, sign));
                    // positions kc = t + (h + 2 c) N/16 and that + N/2
                    o[h + 2 * c] = cadd(a, b);
                    o[h + 2 * c + 8] = csub(a, b);
                }
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = o[q];
        }
        // radix 4 alone: output r of butterfly i lies at t + (i + 4 r) N/16
    }
}

// Threads of one transform wait for each other.  WAVE: they are all of one
// wave, whose LDS accesses keep their order.
template <bool WAVE>
__device__ __forceinline__ void fft_sync()
{
    if constexpr (!WAVE) __syncthreads();
    else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// The whole transform: on entry and on return v[q] is the point t + q N/16
// (the last pass, whatever its radix, leaves them so).  Its LDS entry i is
// buf[fft_pad(i) ST]; every thread that shares the workgroup's LDS calls this
// alike unless WAVE, and buf may still be read by others on entry only if the
// caller synchronises.
template <int N, int ST, bool WAVE, int NS = 1>
__device__ __forceinline__ void fft_run(float2 (&v)[16], int t, const float2* __restrict__ tw,
                                        float sign, float2* buf, bool active = true)
{
    constexpr int R = fft_pass_radix(N, NS);
    if (active) fft_pass<N, NS>(v, t, tw, sign);
    if constexpr (NS * R < N) {
        fft_sync<WAVE>();
        if (active) {
#pragma unroll
            for (int q = 0; q < 16; q++) buf[fft_pad(fft_out<N, NS>(t, q)) * ST] = v[q];
        }
        fft_sync<WAVE>();
        if (active) {
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = buf[fft_pad(t + q * (N / 16)) * ST];
        }
        fft_run<N, ST, WAVE, NS * R>(v, t, tw, sign, buf, active);
    }
}

// Workgroup of row transforms: 256 threads, or those of one transform.
constexpr int fft_row_threads(int n) { return n / 16 > 256 ? n / 16 : 256; }
constexpr int fft_rows(int n) { return fft_row_threads(n) / (n / 16); }   // transforms of it
constexpr bool fft_in_wave(int n) { return n / 16 <= 64; }

// Column transforms of n rows cropped to m that are done in registers.
constexpr bool fft_col_reg_ok(int n, int m)
{
    return fft_reg_ok(n) && n <= 4096 && m >= 64 && (m == n / 2 || m == n / 4 || m == n / 8);
}
constexpr int fft_col_reg_width(int n) { return n <= 256 ? 16 : n <= 1024 ? 8 : 4; }

// Columns that a column transform's workgroup takes, and the width of the
// column blocks in which spectra are stored, [block][row][columns]: a
// workgroup then reads and writes one contiguous range.  Over LDS, two
// buffers of n entries a column: 64 KiB, one column for n > 2048 (128 KiB).
inline int fft_col_width(int n, int m)
{
    if (fft_col_reg_ok(n, m)) return fft_col_reg_width(n);
    return n <= 512 ? 8 : n <= 1024 ? 4 : n <= 2048 ? 2 : 1;
}
