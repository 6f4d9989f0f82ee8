// pg_fftmix_line.hip -- FFT along a strided axis (the x and z passes of the
// oversampled grid) for lengths that are not powers of two.
#include "pg_fftmix.h"

namespace {

// lines per block: consecutive inner indices, so that every global access is
// a run of that many points.  32 (256 bytes) up to length 144, where the block's
// rows stay within 40 KB of LDS (512 threads at most, 640 at 100 and 140), else 16.
template <int N>
constexpr int lpb()
{
    return N <= 144 ? 32 : 16;
}

// Bound by HBM: each point read and written once (zero-padded and cropped
// points never).  Thread (t, j): line j of the block, thread t of the line;
// the LDS rows are an odd multiple of 16 float2 apart, so that the two rows
// that a half-wavefront reads in level 2 lie on different banks.  Forward:
// R1 the multiple of 4, the padded half dropped from level 1.  Adjoint: R2
// the multiple of 4, the cropped half dropped from level 2.
template <int R1, int R2, int SIGN>
__global__ void __launch_bounds__((pgm::line_threads<R1, R2>() * lpb<R1 * R2>()))
    k_line_mix(const float2* __restrict__ src, float2* __restrict__ dst, long long inner_n,
               long long src_os, long long dst_os, const float2* __restrict__ tw)
{
    constexpr int N = R1 * R2;
    constexpr int LPB = lpb<N>();
    constexpr int KST = LPB == 32 ? R2 * 32 + 16 : (R2 | 1) * 16;
    static_assert((SIGN < 0 ? R1 : R2) % 4 == 0, "gridos-2 layout");
    __shared__ float2 lds[R1 * KST];
    const int j = threadIdx.x % LPB, t = threadIdx.x / LPB;
    const long long inner = (long long)blockIdx.x * LPB + j;
    const bool valid = inner < inner_n;
    const float2* s = src + (long long)blockIdx.y * src_os + (valid ? inner : 0);
    float2* d = dst + (long long)blockIdx.y * dst_os + inner;
    float2 v[R1], u[R2];
    if (t < R2) {
#pragma unroll
        for (int m = 0; m < R1; ++m) {
            if (SIGN < 0 && !pgm::half_live<R1>(m)) {
                v[m] = make_float2(0.f, 0.f);
                continue;
            }
            // forward: image row at position t + R2 m; adjoint: ifftshift
            const int q = SIGN < 0 ? t + R2 * ((m + R1 / 4) % R1) : t + R2 * m + N / 2;
            v[m] = s[(long long)(SIGN < 0 || q < N ? q : q - N) * inner_n];
        }
    }
    pgm::line_fft<R1, R2, SIGN>(v, u, t, lds,
                                [j](int k1, int q) { return k1 * KST + q * LPB + j; }, tw);
    if (t >= R1 || !valid) return;
#pragma unroll
    for (int k2 = 0; k2 < R2; ++k2) {
        if (SIGN < 0) {
            const int o = t + R1 * k2 + N / 2;
            d[(long long)(o < N ? o : o - N) * inner_n] = u[k2];
        } else if (pgm::half_live<R2>(k2)) {
            d[(long long)(t + R1 * ((k2 + R2 / 4) % R2)) * inner_n] = u[k2];
        }
    }
}

template <int R1, int R2, int SIGN>
void launch(const float2* src, float2* dst, long long inner_n, long long src_os, long long dst_os,
            unsigned outer, const float2* tw, hipStream_t s)
{
    constexpr int LPB = lpb<R1 * R2>();
    pg::grid_y_runs(outer, [&](long long o, unsigned n) {
        hipLaunchKernelGGL((k_line_mix<R1, R2, SIGN>),
                           dim3((unsigned)((inner_n + LPB - 1) / LPB), n),
                           dim3(pgm::line_threads<R1, R2>() * LPB), 0, s, src + o * src_os,
                           dst + o * dst_os, inner_n, src_os, dst_os, tw);
    });
}

}  // namespace

namespace pgm {

bool mix_len(int n)
{
    switch (n) {
#define PG_CASE(N, A, B) case N:
        PG_MIX_LENGTHS(PG_CASE)
#undef PG_CASE
        return true;
    }
    return false;
}

bool line(int sign, const float2* src, float2* dst, long long inner_n, long long src_os,
          long long dst_os, int nin, int in_off, int nout, int out_off, unsigned outer,
          const pg::FftPlan1D& p, hipStream_t s)
{
    const int n = p.n;
    const bool gridos2 = sign < 0 ? 2 * nin == n && in_off % n == 3 * n / 4 && nout == n &&
                                        out_off % n == n / 2
                                  : nin == n && in_off % n == n / 2 && 2 * nout == n &&
                                        out_off % n == 3 * n / 4;
    if (!gridos2) return false;
    switch (n) {
#define PG_CASE(N, A, B)                                                                      \
    case N:                                                                                   \
        sign < 0 ? launch<A, B, -1>(src, dst, inner_n, src_os, dst_os, outer, p.tw, s)         \
                 : launch<B, A, 1>(src, dst, inner_n, src_os, dst_os, outer, p.tw, s);         \
        return true;
        PG_MIX_LENGTHS(PG_CASE)
#undef PG_CASE
    }
    return false;
}

}  // namespace pgm
