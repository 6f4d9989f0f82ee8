// pg_fftmix_adj.hip -- the adjoint y pass of the oversampled grid (IFFT, crop
// and image weights) for lengths that are not powers of two.
#include <algorithm>

#include "pg_fftmix.h"

namespace {

// lines (columns x segments) of a block
constexpr int kPostLines = 8;

// The adjoint tail of image column col and coil c: for every segment l the
// IFFT along y of column col of grid c L + l (ifftshift on load), the Ny
// cropped rows times WoH_l, summed over l; then dap and conj(S_c).  A block
// holds npc columns x ng groups of a line's threads; group g takes the
// segments g, g + ng, ..., and the groups' sums are added in group order
// through LDS.  R2 is the multiple of 4: a thread's cropped outputs are whole
// entries, so half of level 2 and of the weights drop out and a thread's
// running sums are R2 / 2 points.  Bound by the read of T.
template <int R1, int R2>
__global__ void __launch_bounds__((pgm::line_threads<R1, R2>() * kPostLines))
    k_adj_post_mix(const float2* __restrict__ T, const float2* __restrict__ S,
                   const float2* __restrict__ WoH, const float* __restrict__ dap, int ncol, int L,
                   int npc, int ng, const float2* __restrict__ tw, float2* __restrict__ out,
                   long long out_cstride)
{
    constexpr int N = R1 * R2, Ny = N / 2, TL = pgm::line_threads<R1, R2>();
    constexpr int P = pgm::row_pitch<R2>();
    constexpr int H = R2 / 2;  // image rows per thread: y = t + R1 i
    static_assert(R2 % 4 == 0, "gridos-2 layout");
    __shared__ float2 lds[kPostLines * R1 * P];
    const int t = threadIdx.x % TL, ln = threadIdx.x / TL;
    const int g = ln / npc, jl = ln - g * npc;
    const int c = blockIdx.y;
    const int col = blockIdx.x * npc + jl;
    const long long colc = col < ncol ? col : 0;
    const long long nimg = (long long)ncol * Ny;
    float2 acc[H];
#pragma unroll
    for (int i = 0; i < H; ++i) acc[i] = make_float2(0.f, 0.f);
    float2* my = lds + ln * R1 * P;
    for (int l0 = 0; l0 < L; l0 += ng) {
        const int l = l0 + g;
        const bool live = l < L;
        float2 v[R1], u[R2];
        if (t < R2) {
            const float2* src = T + (((long long)c * L + (live ? l : 0)) * ncol + colc) * N;
#pragma unroll
            for (int m = 0; m < R1; ++m) {
                const int p = t + R2 * m + N / 2;
                v[m] = src[p < N ? p : p - N];
            }
        }
        pgm::line_fft<R1, R2, 1>(v, u, t, my, [](int k1, int q) { return k1 * P + q; }, tw);
        if (t < R1 && live) {
            if (WoH) {
                const float2* Wl = WoH + l * nimg + colc * Ny + t;
                float2 w[H];
#pragma unroll
                for (int i = 0; i < H; ++i) w[i] = Wl[R1 * i];
#pragma unroll
                for (int i = 0; i < H; ++i) {
                    const float2 q = pgf::cmul(u[(i + 3 * R2 / 4) % R2], w[i]);
                    acc[i].x += q.x;
                    acc[i].y += q.y;
                }
            } else {
#pragma unroll
                for (int i = 0; i < H; ++i) {
                    acc[i].x += u[(i + 3 * R2 / 4) % R2].x;
                    acc[i].y += u[(i + 3 * R2 / 4) % R2].y;
                }
            }
        }
        __syncthreads();  // the next segment's exchange reuses the rows
    }
    float2* red = lds;  // [line][row]: Ny <= R1 * P slots per line
    if (t < R1) {
#pragma unroll
        for (int i = 0; i < H; ++i) red[ln * Ny + t + R1 * i] = acc[i];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < npc * Ny; e += blockDim.x) {
        const int jj = e / Ny, y = e - jj * Ny;
        const int cc = blockIdx.x * npc + jj;
        if (cc >= ncol) continue;
        float2 sum = red[jj * Ny + y];
        for (int k = 1; k < ng; ++k) {
            const float2 a = red[(k * npc + jj) * Ny + y];
            sum.x += a.x;
            sum.y += a.y;
        }
        const long long nidx = (long long)y + (long long)cc * Ny;
        if (dap) {
            const float d = dap[nidx];
            sum = make_float2(sum.x * d, sum.y * d);
        }
        if (S) {
            float2 sc = S[(long long)c * nimg + nidx];
            sc.y = -sc.y;
            sum = pgf::cmul(sum, sc);
        }
        out[c * out_cstride + nidx] = sum;
    }
}

template <int R1, int R2>
void launch(const float2* T, const float2* S, const float2* WoH, const float* dap, int ncol, int nc,
            int L, const float2* tw, float2* out, long long out_cstride, hipStream_t s)
{
    constexpr int TL = pgm::line_threads<R1, R2>(), NL = kPostLines;
    // as many segments in flight as a block holds, in equal rounds (12
    // segments: 6 + 6), then columns up to two wavefronts
    const int rounds = (L + NL - 1) / NL;
    const int ng = (L + rounds - 1) / rounds;
    const int npc = std::max(1, std::min(NL / ng, 128 / (ng * TL)));
    // (planes of a stack: there may be more than a grid dimension holds)
    pg::grid_y_runs(nc, [&](long long o, unsigned n) {
        hipLaunchKernelGGL((k_adj_post_mix<R1, R2>), dim3((ncol + npc - 1) / npc, n),
                           dim3(TL * npc * ng), 0, s, T + o * L * ncol * (R1 * R2),
                           S ? S + o * ncol * (R1 * R2 / 2) : S, WoH, dap, ncol, L, npc, ng, tw,
                           out + o * out_cstride, out_cstride);
    });
}

}  // namespace

namespace pgm {

void adj_post(const float2* T, const float2* S, const float2* WoH, const float* dap, int ncol,
              int nc, int L, const pg::FftPlan1D& p, float2* out, long long out_cstride,
              hipStream_t s)
{
    switch (p.n) {
#define PG_CASE(N, A, B)                                                                  \
    case N:                                                                               \
        launch<B, A>(T, S, WoH, dap, ncol, nc, L, p.tw, out, out_cstride, s);             \
        return;
        PG_MIX_LENGTHS(PG_CASE)
#undef PG_CASE
    }
    throw pg::Error{PG_ERR_STATE, "no register FFT for this length"};
}

}  // namespace pgm
