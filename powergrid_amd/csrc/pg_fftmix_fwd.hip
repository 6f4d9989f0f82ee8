// pg_fftmix_fwd.hip -- the forward y pass of the oversampled grid (image
// weights, zero padding and FFT) for lengths that are not powers of two.
#include "pg_fftmix.h"

namespace {

// image columns per block of the forward pass, about 256 threads
template <int R1, int R2>
constexpr int col_lpb()
{
    return 256 / pgm::line_threads<R1, R2>();
}

// v = dap Wo_l S_c x of image column col, zero-padded to N (image row y at
// (y + 3N/4) % N), FFT along y, entry k to (k + N/2) % N of T.  Every load
// goes to an in-bounds address whether the column exists or not, so that all
// loads of a thread are in flight together.  Bound by the write of T.
template <int R1, int R2>
__global__ void __launch_bounds__((pgm::line_threads<R1, R2>() * col_lpb<R1, R2>()))
    k_fwd_col_mix(const float2* __restrict__ img, long long img_cstride,
                  const float2* __restrict__ S, const float2* __restrict__ Wo,
                  const float* __restrict__ dap, int ncol, int L, const float2* __restrict__ tw,
                  float2* __restrict__ T)
{
    constexpr int N = R1 * R2, Ny = N / 2, TL = pgm::line_threads<R1, R2>();
    constexpr int P = pgm::row_pitch<R2>();
    constexpr int H = R1 / 2;  // image rows per thread: y = t + R2 i
    static_assert(R1 % 4 == 0, "gridos-2 layout");
    __shared__ float2 lds[col_lpb<R1, R2>() * R1 * P];
    const int t = threadIdx.x % TL, jl = threadIdx.x / TL;
    const int b = blockIdx.y;
    const int c = b / L, l = b - c * L;
    const int col = blockIdx.x * (blockDim.x / TL) + jl;
    const bool valid = col < ncol;
    const long long nimg = (long long)ncol * Ny;
    const long long ofs = (long long)(valid ? col : 0) * Ny + t;
    float2 v[R1], u[R2];
    if (t < R2) {
        float2 x[H];
        const float2* im = img + c * img_cstride + ofs;
#pragma unroll
        for (int i = 0; i < H; ++i) x[i] = im[R2 * i];
        if (S) {
            const float2* q = S + c * nimg + ofs;
            float2 w[H];
#pragma unroll
            for (int i = 0; i < H; ++i) w[i] = q[R2 * i];
#pragma unroll
            for (int i = 0; i < H; ++i) x[i] = pgf::cmul(w[i], x[i]);
        }
        if (Wo) {
            const float2* q = Wo + l * nimg + ofs;
            float2 w[H];
#pragma unroll
            for (int i = 0; i < H; ++i) w[i] = q[R2 * i];
#pragma unroll
            for (int i = 0; i < H; ++i) x[i] = pgf::cmul(w[i], x[i]);
        }
        if (dap) {
            const float* q = dap + ofs;
            float w[H];
#pragma unroll
            for (int i = 0; i < H; ++i) w[i] = q[R2 * i];
#pragma unroll
            for (int i = 0; i < H; ++i) x[i] = make_float2(x[i].x * w[i], x[i].y * w[i]);
        }
#pragma unroll
        for (int m = 0; m < R1; ++m)
            v[m] = pgm::half_live<R1>(m) ? x[(m + R1 / 4) % R1] : make_float2(0.f, 0.f);
    }
    float2* my = lds + jl * R1 * P;
    pgm::line_fft<R1, R2, -1>(v, u, t, my, [](int k1, int q) { return k1 * P + q; }, tw);
    if (t >= R1 || !valid) return;
    float2* dst = T + ((long long)b * ncol + col) * N;
#pragma unroll
    for (int k2 = 0; k2 < R2; ++k2) {
        const int o = t + R1 * k2 + N / 2;
        dst[o < N ? o : o - N] = u[k2];
    }
}

template <int R1, int R2>
void launch(const float2* img, long long img_cstride, const float2* S, const float2* Wo,
            const float* dap, int ncol, int B, int L, const float2* tw, float2* T, hipStream_t s)
{
    constexpr int TL = pgm::line_threads<R1, R2>();
    // fewer columns per block where the launch would leave compute units idle
    int lpb = col_lpb<R1, R2>();
    while (lpb > 2 && (long long)((ncol + lpb - 1) / lpb) * B < 512) lpb = (lpb + 1) / 2;
    if (L == 1 && !S) {
        // (planes of a stack: there may be more than a grid dimension holds)
        pg::grid_y_runs(B, [&](long long o, unsigned n) {
            hipLaunchKernelGGL((k_fwd_col_mix<R1, R2>), dim3((ncol + lpb - 1) / lpb, n),
                               dim3(TL * lpb), 0, s, img + o * img_cstride, img_cstride, S, Wo, dap,
                               ncol, L, tw, T + o * ncol * (R1 * R2));
        });
        return;
    }
    hipLaunchKernelGGL((k_fwd_col_mix<R1, R2>), dim3((ncol + lpb - 1) / lpb, B), dim3(TL * lpb), 0,
                       s, img, img_cstride, S, Wo, dap, ncol, L, tw, T);
}

}  // namespace

namespace pgm {

void fwd_col(const float2* img, long long img_cstride, const float2* S, const float2* Wo,
             const float* dap, int ncol, int B, int L, const pg::FftPlan1D& p, float2* T,
             hipStream_t s)
{
    switch (p.n) {
#define PG_CASE(N, A, B_)                                                             \
    case N:                                                                           \
        launch<A, B_>(img, img_cstride, S, Wo, dap, ncol, B, L, p.tw, T, s);          \
        return;
        PG_MIX_LENGTHS(PG_CASE)
#undef PG_CASE
    }
    throw pg::Error{PG_ERR_STATE, "no register FFT for this length"};
}

}  // namespace pgm
