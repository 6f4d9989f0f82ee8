// pg_fftmix.h -- register FFT passes for grid lengths that are not powers of
// two (their prime factors at most 13), gfx950.
//
// A line of length N = R1*R2 is transformed in two levels with one exchange
// through LDS, as pg_fftreg.h does for powers of two, with any pair of the
// register DFTs below:
//   1. thread t < R2 holds v[m] = x[t + R2*m], m < R1, does a length-R1 DFT
//      in registers and multiplies entry k1 by w_N^(t*k1);
//   2. thread k1 < R1 does the length-R2 DFT over t and holds X[k1 + R1*k2].
// The LDS Stockham form runs five or six radix-2/3/4/5 stages on such a
// length, each with a barrier, runtime divisions and an LDS round trip; here
// every index is a compile-time function of (t, m).  Measured on 384 grids of
// 384^2 (192^2 image, 32 coils, 12 segments; each x pass moves 680 MB): x
// passes 539 and 629 -> 144 and 167 us (4.7 and 4.1 TB/s, the rate of a large
// copy), forward y pass 206 -> 88 us, adjoint y pass with the segment sum
// 330 -> 87 us.
#pragma once

#include "pg_fftreg.h"

namespace pgm {

// ------------------------------------------------------- register DFTs --
// R = A * B with the length-A transforms first
template <int R>
constexpr int split_a()
{
    return R == 6 ? 2 : R == 9 ? 3 : R == 10 ? 2 : R == 12 ? 4 : R == 14 ? 2 : R == 15 ? 3
         : R == 18 ? 2 : R == 20 ? 4 : R == 22 ? 2 : R == 24 ? 8 : R == 26 ? 2 : R == 28 ? 4 : 1;
}

// odd prime R: with s_j = v_j + v_(R-j), d_j = v_j - v_(R-j),
//   X_k     = v_0 + sum_j cos(2 pi j k / R) s_j + SIGN i sum_j sin(2 pi j k / R) d_j
//   X_(R-k) = the same with the second sum subtracted
template <int R, int SIGN>
__host__ __device__ __forceinline__ void prime_dft(float2 (&v)[R])
{
    constexpr pgf::Tw<R> tw{};  // exp(-2 pi i k / R)
    constexpr int H = (R - 1) / 2;
    float2 s[H], d[H];
#pragma unroll
    for (int j = 0; j < H; ++j) {
        s[j] = make_float2(v[j + 1].x + v[R - 1 - j].x, v[j + 1].y + v[R - 1 - j].y);
        d[j] = make_float2(v[j + 1].x - v[R - 1 - j].x, v[j + 1].y - v[R - 1 - j].y);
    }
    const float2 v0 = v[0];
#pragma unroll
    for (int j = 0; j < H; ++j) v[0] = make_float2(v[0].x + s[j].x, v[0].y + s[j].y);
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        float2 c = v0, e = make_float2(0.f, 0.f);
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            const int q = (j * k) % R;
            c.x += tw.c[q] * s[j - 1].x;
            c.y += tw.c[q] * s[j - 1].y;
            e.x -= tw.s[q] * d[j - 1].x;
            e.y -= tw.s[q] * d[j - 1].y;
        }
        // SIGN i e
        const float2 u = SIGN > 0 ? make_float2(-e.y, e.x) : make_float2(e.y, -e.x);
        v[k] = make_float2(c.x + u.x, c.y + u.y);
        v[R - k] = make_float2(c.x - u.x, c.y - u.y);
    }
}

// in-register DFT of length R, natural order in and out
template <int R, int SIGN>
__host__ __device__ __forceinline__ void dft(float2 (&v)[R])
{
    if constexpr (R == 1) {
        return;
    } else if constexpr ((R & (R - 1)) == 0) {
        pgf::reg_dft<R, SIGN>(v);
    } else if constexpr (split_a<R>() == 1) {
        prime_dft<R, SIGN>(v);
    } else {
        // n = b + B a, k = k1 + A k2
        constexpr int A = split_a<R>(), B = R / A;
        constexpr pgf::Tw<R> tw{};
        float2 w[R];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            float2 u[A];
#pragma unroll
            for (int a = 0; a < A; ++a) u[a] = v[b + B * a];
            dft<A, SIGN>(u);
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) w[b + B * k1] = pgf::twid<SIGN, R>(u[k1], b * k1, tw);
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            float2 u[B];
#pragma unroll
            for (int b = 0; b < B; ++b) u[b] = w[b + B * k1];
            dft<B, SIGN>(u);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = u[k2];
        }
    }
}

// The supported lengths and their factors, f(N, A, B): A a multiple of 4 (the
// zero-padded or cropped half of a gridos-2 line is then whole entries of the
// length-A level, see half_live), both near sqrt(N) and at most 28, so that a
// thread holds at most 56 floats of the line.  The lengths are those of images
// of even size up to 240 with factors like these; 324, 420, 440 and longer ones
// that have such factors (500 ... 784) are not listed and take the Stockham form.  The
// passes serve the gridos-2
// layout alone: image row i of N/2 at position (i + 3N/4) mod N.
#define PG_MIX_LENGTHS(f)                                                                        \
    f(20, 4, 5) f(24, 8, 3) f(28, 4, 7) f(36, 12, 3) f(40, 8, 5) f(44, 4, 11) f(48, 8, 6)       \
    f(52, 4, 13) f(56, 8, 7) f(60, 12, 5)                                                        \
    f(72, 12, 6) f(80, 16, 5) f(84, 12, 7) f(88, 8, 11) f(96, 12, 8) f(100, 20, 5)              \
    f(104, 8, 13) f(108, 12, 9) f(112, 16, 7) f(120, 12, 10) f(132, 12, 11) f(140, 20, 7)       \
    f(144, 12, 12) f(156, 12, 13) f(160, 16, 10) f(168, 24, 7) f(176, 16, 11) f(180, 20, 9)     \
    f(192, 16, 12) f(196, 28, 7) f(200, 20, 10) f(208, 16, 13) f(216, 24, 9) f(220, 20, 11)     \
    f(224, 16, 14) f(240, 16, 15) f(252, 28, 9) f(260, 20, 13) f(264, 24, 11) f(280, 20, 14)    \
    f(288, 24, 12) f(300, 20, 15) f(308, 28, 11) f(312, 24, 13) f(320, 20, 16) f(336, 24, 14)   \
    f(352, 16, 22) f(360, 24, 15) f(364, 28, 13) f(384, 24, 16) f(392, 28, 14) f(400, 20, 20)   \
    f(416, 16, 26) f(432, 24, 18) f(448, 28, 16) f(480, 24, 20)

template <int R1, int R2>
constexpr int line_threads()
{
    return R1 > R2 ? R1 : R2;
}

// LDS slots of a line in the y passes: entry k1 of thread q at k1 * P + q, P odd, so that
// both the writes (consecutive q) and the reads (consecutive k1) are spread
// over the banks
template <int R2>
constexpr int row_pitch()
{
    return R2 | 1;
}

// whether entry m of a level of length R (a multiple of 4) is an image row of
// the gridos-2 layout, for every thread
template <int R>
constexpr bool half_live(int m)
{
    return m < R / 4 || m >= 3 * R / 4;
}

// levels 1 and 2 for one line: `at(k1, q)` is the LDS slot of entry k1 of
// thread q; v holds x[t + R2 m] on entry (t < R2), u X[t + R1 k2] on return
// (t < R1)
template <int R1, int R2, int SIGN, class At>
__device__ __forceinline__ void line_fft(float2 (&v)[R1], float2 (&u)[R2], int t, float2* lds, At at,
                                         const float2* __restrict__ tw)
{
    if (t < R2) {
        dft<R1, SIGN>(v);
#pragma unroll
        for (int k1 = 1; k1 < R1; ++k1) {
            float2 w = tw[t * k1];
            if (SIGN > 0) w.y = -w.y;
            v[k1] = pgf::cmul(v[k1], w);
        }
#pragma unroll
        for (int k1 = 0; k1 < R1; ++k1) lds[at(k1, t)] = v[k1];
    }
    __syncthreads();
    if (t < R1) {
#pragma unroll
        for (int q = 0; q < R2; ++q) u[q] = lds[at(t, q)];
        dft<R2, SIGN>(u);
    }
}

}  // namespace pgm

// ---------------------------------------------------------- launchers ----
#include "pg_internal.h"
namespace pgm {

// whether a length has these kernels
bool mix_len(int n);

// FFT along a strided axis, the arguments of line_fft_any (pg_fft.hip).
// Returns false, having launched nothing, unless the length has a kernel and
// the layout is that of gridos 2 (forward: half the inputs, adjoint: half the
// outputs are image rows).
bool line(int sign, const float2* src, float2* dst, long long inner_n, long long src_os,
          long long dst_os, int nin, int in_off, int nout, int out_off, unsigned outer,
          const pg::FftPlan1D& p, hipStream_t s);

// whether the y passes of an image of Ny rows on a grid line of n run here
inline bool col_ok(int n, int Ny, int offY)
{
    return mix_len(n) && 2 * Ny == n && offY == n / 4;
}

// image weights + zero padding + FFT along y of ncol image columns of each of
// B = nc*L grids into T (S, Wo and dap may be null: not applied)
void fwd_col(const float2* img, long long img_cstride, const float2* S, const float2* Wo,
             const float* dap, int ncol, int B, int L, const pg::FftPlan1D& p, float2* T,
             hipStream_t s);

// IFFT along y, crop, deapodization, WoH, sum over the segments, conj(S):
// the arguments of the adjoint tail (S, WoH and dap may be null)
void adj_post(const float2* T, const float2* S, const float2* WoH, const float* dap, int ncol,
              int nc, int L, const pg::FftPlan1D& p, float2* out, long long out_cstride,
              hipStream_t s);

}  // namespace pgm
