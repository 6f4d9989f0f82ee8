// pg_dft.hip -- exact field-corrected DFT (Gdft, Gdft.cpp:52-136 /
// ftCpu.cpp:94-215), batched over SENSE coils.
//   forward: y_c[i] = sum_j S_c[j] x[j] exp(-i (2 pi k_i . r_j + fm_j t_i))
//   adjoint: x[j]   = sum_c conj(S_c[j]) sum_i y_c[i] exp(+i (...))
// The phase of a (sample, pixel) pair is computed once and used for every
// coil.  Work is split over (output block, input slice); slices are summed
// by a second kernel in a fixed order.
// pcSENSE's shots (pcSENSE.cpp:108-153) run as one launch: the M samples
// are nshot shots of M/nshot, shot-major, and shot s has its own nc maps at
// S + s * s_shot.  Forward sample tiles and adjoint sample slices never
// straddle a shot, so a block applies one shot's maps.
//
// precision 0 -- the reference's arithmetic class (FP32 phase, FP32 trig):
//   the phase is formed in revolutions, p = k.r + fm t / (2 pi), reduced to
//   [-1/2, 1/2] and fed to the hardware v_sin_f32 / v_cos_f32 (which take
//   revolutions); FP32 accumulation.
// precision 1 -- FP64 phase, FP64 sin/cos, FP64 accumulation (the exact
//   NUDFT; used to synthesise data and as an accuracy reference).
// GdftR2 (GdftR2.cpp, ftCpuWithGrads.cpp:98-212) multiplies every pair by
//   b = sinc(kx/Nx + Gx t) sinc(ky/Ny + Gy t) sinc(kz/Nz + Gz t),
//   sinc(x) = sin(pi x)/(pi x) (1 below 1e-4), with the field-map difference
//   maps G staged beside the pixel coordinates.
#include "pg_dft.h"
#include "pg_fftreg.h"

#include <mutex>

namespace {

// partial sums of pg_dft_apply_static: every element a launch reads was
// written earlier in the same launch sequence, so nothing is cleared
constexpr size_t kScratchElems = (size_t)8 << 20;  // 8M float2 = 64 MiB
__device__ __align__(256) float2 scratch[kScratchElems];

constexpr int kT = 64;  // threads per block (one wavefront) = tile width

// sin(pi x)/(pi x) in FP32 with the hardware sine (which takes revolutions:
// sin(pi x) = sin(2 pi (x/2)), reduced to [-1/2, 1/2] turns first)
__device__ __forceinline__ float sinc_f(float x)
{
    if (fabsf(x) < 1e-4f) return 1.0f;
    float r = 0.5f * x;
    r = r - rintf(r);
    return __builtin_amdgcn_sinf(r) / (3.14159265358979f * x);
}

__device__ __forceinline__ double sinc_d(double x)
{
    if (fabs(x) < 1e-4) return 1.0;
    return sin(M_PI * x) / (M_PI * x);
}

struct R2Args {
    const float *gx, *gy, *gz;
    float inx, iny, inz;  // 1/Nx, 1/Ny, 1/Nz
};

// FP64 phase, trig and sums (precision 1): one wavefront per 64 outputs and
// input slice, the inputs staged in LDS; bound by the FP64 sine and cosine.
template <int NCB, bool R2>
__global__ void __launch_bounds__(kT) k_gdft_fwd(
    const float* __restrict__ kx, const float* __restrict__ ky, const float* __restrict__ kz,
    const float* __restrict__ t, const float* __restrict__ ix, const float* __restrict__ iy,
    const float* __restrict__ iz, const float* __restrict__ fm, const float2* __restrict__ x,
    const float2* __restrict__ S, int nc, int M, int N, int slice_len, int shot_len,
    long long s_shot, float2* __restrict__ part, R2Args r2)
{
    __shared__ float s_r[kT][4];
    __shared__ float s_g[R2 ? kT : 1][3];
    __shared__ float2 s_v[kT][NCB];
    // ceil(shot_len / kT) tiles per shot
    const int tps = (shot_len + kT - 1) / kT;
    const int sh = blockIdx.x / tps;
    const int il = (blockIdx.x - sh * tps) * kT + threadIdx.x;
    const bool live = il < shot_len;
    const int i = sh * shot_len + il;
    if (S) S += sh * s_shot;
    const int c0 = blockIdx.z * NCB;
    const int j0 = blockIdx.y * slice_len;
    const int j1 = min(N, j0 + slice_len);
    float ki[3] = {0, 0, 0};
    float ti = 0;
    if (live) {
        ki[0] = kx[i];
        ki[1] = ky[i];
        ki[2] = kz[i];
        ti = t[i];
    }
    double ar[NCB], ai[NCB];
#pragma unroll
    for (int c = 0; c < NCB; ++c) ar[c] = ai[c] = 0.0;

    for (int jb = j0; jb < j1; jb += kT) {
        __syncthreads();
        const int j = jb + threadIdx.x;
        if (j < j1) {
            s_r[threadIdx.x][0] = ix[j];
            s_r[threadIdx.x][1] = iy[j];
            s_r[threadIdx.x][2] = iz[j];
            s_r[threadIdx.x][3] = fm[j];
            if (R2) {
                s_g[threadIdx.x][0] = r2.gx[j];
                s_g[threadIdx.x][1] = r2.gy[j];
                s_g[threadIdx.x][2] = r2.gz[j];
            }
            const float2 xv = x[j];
#pragma unroll
            for (int c = 0; c < NCB; ++c) {
                float2 v = xv;
                if (S && c0 + c < nc) {
                    const float2 s = S[(long long)(c0 + c) * N + j];
                    v = make_float2(s.x * xv.x - s.y * xv.y, s.x * xv.y + s.y * xv.x);
                }
                s_v[threadIdx.x][c] = v;
            }
        }
        __syncthreads();
        const int cnt = min(kT, j1 - jb);
        for (int q = 0; q < cnt; ++q) {
            const double ph = 2.0 * M_PI * ((double)ki[0] * s_r[q][0] + (double)ki[1] * s_r[q][1] +
                                            (double)ki[2] * s_r[q][2]) +
                              (double)s_r[q][3] * ti;
            double sd, cd;
            sincos(ph, &sd, &cd);
            if (R2) {
                const double b = sinc_d((double)ki[0] * r2.inx + (double)s_g[q][0] * ti) *
                                 sinc_d((double)ki[1] * r2.iny + (double)s_g[q][1] * ti) *
                                 sinc_d((double)ki[2] * r2.inz + (double)s_g[q][2] * ti);
                sd *= b;
                cd *= b;
            }
#pragma unroll
            for (int c = 0; c < NCB; ++c) {
                const float2 v = s_v[q][c];
                ar[c] += cd * v.x + sd * v.y;
                ai[c] += -sd * v.x + cd * v.y;
            }
        }
    }
    if (live) {
#pragma unroll
        for (int c = 0; c < NCB; ++c) {
            if (c0 + c >= nc) break;
            part[((long long)blockIdx.y * nc + c0 + c) * M + i] =
                make_float2((float)ar[c], (float)ai[c]);
        }
    }
}

template <int NCB, bool R2>
__global__ void __launch_bounds__(kT) k_gdft_adj(
    const float* __restrict__ kx, const float* __restrict__ ky, const float* __restrict__ kz,
    const float* __restrict__ t, const float* __restrict__ ix, const float* __restrict__ iy,
    const float* __restrict__ iz, const float* __restrict__ fm, const float2* __restrict__ y,
    long long ystride, const float2* __restrict__ S, int nc, int M, int N, int slice_len,
    int shot_len, long long s_shot, float2* __restrict__ part, R2Args r2)
{
    __shared__ float s_k[kT][4];
    __shared__ float2 s_v[kT][NCB];
    const int j = blockIdx.x * kT + threadIdx.x;
    // gridDim.y / nshot slices per shot, each within its shot
    const int sps = (int)gridDim.y / (M / shot_len);
    const int sh = blockIdx.y / sps;
    const int i0 = sh * shot_len + (blockIdx.y - sh * sps) * slice_len;
    const int i1 = min(sh * shot_len + shot_len, i0 + slice_len);
    if (S) S += sh * s_shot;
    float rj[3] = {0, 0, 0};
    float fj = 0;
    float gj[3] = {0, 0, 0};
    if (j < N) {
        rj[0] = ix[j];
        rj[1] = iy[j];
        rj[2] = iz[j];
        fj = fm[j];
        if (R2) {
            gj[0] = r2.gx[j];
            gj[1] = r2.gy[j];
            gj[2] = r2.gz[j];
        }
    }
    double xr = 0, xi = 0;
    for (int c0 = 0; c0 < nc; c0 += NCB) {
        double ar[NCB], ai[NCB];
#pragma unroll
        for (int c = 0; c < NCB; ++c) ar[c] = ai[c] = 0;
        for (int ib = i0; ib < i1; ib += kT) {
            __syncthreads();
            const int i = ib + threadIdx.x;
            if (i < i1) {
                s_k[threadIdx.x][0] = kx[i];
                s_k[threadIdx.x][1] = ky[i];
                s_k[threadIdx.x][2] = kz[i];
                s_k[threadIdx.x][3] = t[i];
#pragma unroll
                for (int c = 0; c < NCB; ++c)
                    s_v[threadIdx.x][c] = (c0 + c < nc) ? y[(long long)(c0 + c) * ystride + i]
                                                        : make_float2(0.f, 0.f);
            }
            __syncthreads();
            const int cnt = min(kT, i1 - ib);
            for (int q = 0; q < cnt; ++q) {
                const double ph = 2.0 * M_PI * ((double)s_k[q][0] * rj[0] + (double)s_k[q][1] * rj[1] +
                                                (double)s_k[q][2] * rj[2]) +
                                  (double)fj * s_k[q][3];
                double sd, cd;
                sincos(ph, &sd, &cd);
                if (R2) {
                    const double tq = s_k[q][3];
                    const double b = sinc_d((double)s_k[q][0] * r2.inx + (double)gj[0] * tq) *
                                     sinc_d((double)s_k[q][1] * r2.iny + (double)gj[1] * tq) *
                                     sinc_d((double)s_k[q][2] * r2.inz + (double)gj[2] * tq);
                    sd *= b;
                    cd *= b;
                }
#pragma unroll
                for (int c = 0; c < NCB; ++c) {
                    const float2 v = s_v[q][c];
                    ar[c] += cd * v.x - sd * v.y;
                    ai[c] += sd * v.x + cd * v.y;
                }
            }
        }
        if (j < N) {
#pragma unroll
            for (int c = 0; c < NCB; ++c) {
                if (c0 + c >= nc) break;
                double vr = ar[c], vi = ai[c];
                if (S) {
                    const float2 s = S[(long long)(c0 + c) * N + j];
                    const double tr = vr * s.x + vi * s.y;  // v * conj(s)
                    const double ti = vi * s.x - vr * s.y;
                    vr = tr;
                    vi = ti;
                }
                xr += vr;
                xi += vi;
            }
        }
    }
    if (j < N) part[(long long)blockIdx.y * N + j] = make_float2((float)xr, (float)xi);
}

// ------------------------------------------------ FP32 on the matrix cores --
// Both directions are products: with the phase p of (output o, input q),
//   forward  Y[o][2c], Y[o][2c+1] = sum_q cos(p) (vr, vi)_qc + sin(p) (vi, -vr)_qc
//   adjoint  the same with (-vi, vr)
// over the inputs' values v_qc (S_c x, or y_c).  A wavefront takes 64 outputs
// and 4 inputs a step: lane (i, k) = (lane % 16, lane / 16) forms the phase,
// sine and cosine of output 16 t + i and input k for each of the four output
// tiles t, which is the A operand A[i][k] of v_mfma_f32_16x16x4f32; column j
// of the B operand B[k][j] (lane j + 16 k) is float j of input k's row of
// 16 CT values (8 CT coils, re and im), the second one its neighbour's with
// the sign.  The phase arithmetic is that of precision 0
// above (FP32, reduced to [-1/2, 1/2] revolutions, v_sin and v_cos) and the
// sums are FP32.  Per 64 pairs: 16 vector instructions, sine and cosine
// at a quarter of the rate (88 clocks, the bound), beside 2 CT products of 32
// clocks on the matrix cores; forming the sums on the vector units took 32 more
// instructions and 5 LDS broadcasts for 8 coils.
// The four wavefronts of a block take a quarter of the input slice each and
// are summed through LDS in order, so a quarter of the partial sums reach
// memory.  4096 samples x 4096 voxels, 8 coils: forward 34 -> 20.5 us, adjoint
// 29 -> 20.5 us (9.4 of it the vector instructions, the rest launch, staging
// and the wavefronts' sum), and the slice sums 18.5 -> 4.5 us each.
typedef float pgd_f4 __attribute__((ext_vector_type(4)));
constexpr int kMW = 4;       // wavefronts per block
constexpr int kMChunk = 64;  // inputs staged per wavefront at a time

template <int CT>
struct MfmaLds {
    union {
        struct {
            float v[kMW][kMChunk][16 * CT + 4];
            float4 r[kMW][kMChunk];
            float3 g[kMW][kMChunk];
        } in;
        float sum[kMW][64][16 * CT + 1];
    };
};

// the sums over inputs [q0, q1) (this wavefront's share) for outputs with
// coordinates co[t] (+ gradient maps go[t] of an R2 adjoint): acc[t][n], tile
// t, float tile n.  load(q, row, rr, gg) stages input q (a lane's own).
template <int CT, bool R2, bool ADJ, class Load>
__device__ __forceinline__ void dft_products(const float4 (&co)[4], const float3 (&go)[4], int q0,
                                             int q1, float (*sv)[16 * CT + 4], float4* sr, float3* sg,
                                             const R2Args& r2, Load load, pgd_f4 (&acc)[4][CT])
{
    const int lane = threadIdx.x & 63, j = lane & 15, k = lane >> 4;
    // the second product's column: its neighbour's value, negated for the im
    // (forward) or re (adjoint) columns
    const int flip = ((j & 1) != 0) != ADJ ? (int)0x80000000u : 0;
    for (int qb = q0; qb < q1; qb += kMChunk) {
        const int n = min(kMChunk, q1 - qb);
        load(qb + lane, lane < n, sv[lane], sr[lane], sg[lane]);
        pgf::wave_lds_sync();
#pragma unroll 2
        for (int s = 0; s < n; s += 4) {
            const float4 r = sr[s + k];
            float3 gq = make_float3(0.f, 0.f, 0.f);
            if (R2 && !ADJ) gq = sg[s + k];
            float b[CT], bx[CT];
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                b[c] = sv[s + k][16 * c + j];
                const int nb = __builtin_amdgcn_update_dpp(0, __float_as_int(b[c]), 0xB1, 0xF, 0xF,
                                                           false);  // quad_perm [1,0,3,2]
                bx[c] = __int_as_float(nb ^ flip);
            }
            float cs[4], sn[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                float p = co[t].x * r.x + co[t].y * r.y + co[t].z * r.z + r.w * co[t].w;
                p = p - rintf(p);
                sn[t] = __builtin_amdgcn_sinf(p);
                cs[t] = __builtin_amdgcn_cosf(p);
                if (R2) {
                    // k and t of the sample, the maps of the voxel
                    const float4 kk = ADJ ? r : co[t];
                    const float3 gg = ADJ ? go[t] : gq;
                    const float f = sinc_f(kk.x * r2.inx + gg.x * kk.w) *
                                    sinc_f(kk.y * r2.iny + gg.y * kk.w) *
                                    sinc_f(kk.z * r2.inz + gg.z * kk.w);
                    sn[t] *= f;
                    cs[t] *= f;
                }
            }
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(cs[t], b[c], acc[t][c], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(sn[t], bx[c], acc[t][c], 0, 0, 0);
        }
        pgf::wave_lds_sync();  // the next chunk replaces these inputs
    }
}

// this wavefront's sums to LDS: sum[wave][output][float]
template <int CT>
__device__ __forceinline__ void dft_store(float (*out)[16 * CT + 1], const pgd_f4 (&acc)[4][CT])
{
    const int lane = threadIdx.x & 63, j = lane & 15, k = lane >> 4;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[16 * t + 4 * k + r][16 * c + j] = acc[t][c][r];
}

template <int CT, bool R2>
__global__ void __launch_bounds__(64 * kMW) k_gdft_fwd_mfma(
    const float* __restrict__ kx, const float* __restrict__ ky, const float* __restrict__ kz,
    const float* __restrict__ t, const float* __restrict__ ix, const float* __restrict__ iy,
    const float* __restrict__ iz, const float* __restrict__ fm, const float2* __restrict__ x,
    const float2* __restrict__ S, int nc, int M, int N, int slice_len, int shot_len,
    long long s_shot, float2* __restrict__ part, R2Args r2)
{
    __shared__ MfmaLds<CT> lds;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int tps = (shot_len + 63) / 64;  // output tiles per shot
    const int sh = blockIdx.x / tps;
    const int o0 = (blockIdx.x - sh * tps) * 64;
    if (S) S += sh * s_shot;
    const int c0 = blockIdx.z * 8 * CT;
    float4 co[4];
    float3 go[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = sh * shot_len + min(o0 + 16 * u + (lane & 15), shot_len - 1);
        co[u] = make_float4(kx[i], ky[i], kz[i], t[i]);
        go[u] = make_float3(0.f, 0.f, 0.f);
    }
    pgd_f4 acc[4][CT];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[u][c] = pgd_f4{0.f, 0.f, 0.f, 0.f};
    // this wavefront's quarter of the slice, in whole steps of 4 inputs
    const int j0 = blockIdx.y * slice_len, j1 = min(N, j0 + slice_len);
    const int quarter = ((j1 - j0 + 4 * kMW - 1) / (4 * kMW)) * 4;
    const int q0 = min(j1, j0 + wv * quarter), q1 = min(j1, q0 + quarter);
    dft_products<CT, R2, false>(
        co, go, q0, q1, lds.in.v[wv], lds.in.r[wv], lds.in.g[wv], r2,
        [&](int q, bool ok, float* row, float4& rr, float3& gg) {
            const int qc = ok ? q : 0;
            const float2 xv = x[qc];
            rr = make_float4(ix[qc], iy[qc], iz[qc], (float)((double)fm[qc] / (2.0 * M_PI)));
            if (R2) gg = make_float3(r2.gx[qc], r2.gy[qc], r2.gz[qc]);
            float2 sm[8 * CT];
            if (S) {
#pragma unroll
                for (int c = 0; c < 8 * CT; ++c)
                    sm[c] = S[(long long)min(c0 + c, nc - 1) * N + qc];
            }
#pragma unroll
            for (int c = 0; c < 8 * CT; ++c) {
                float2 v = xv;
                if (S)
                    v = make_float2(sm[c].x * xv.x - sm[c].y * xv.y, sm[c].x * xv.y + sm[c].y * xv.x);
                const bool on = ok && c0 + c < nc;
                row[2 * c] = on ? v.x : 0.f;
                row[2 * c + 1] = on ? v.y : 0.f;
            }
        },
        acc);
    __syncthreads();
    dft_store<CT>(lds.sum[wv], acc);
    __syncthreads();
    const int o = o0 + lane;
    if (o >= shot_len) return;
#pragma unroll
    for (int u = 0; u < 2 * CT; ++u) {
        const int c = wv * 2 * CT + u;
        if (c0 + c >= nc) break;
        float2 a = make_float2(lds.sum[0][lane][2 * c], lds.sum[0][lane][2 * c + 1]);
#pragma unroll
        for (int w = 1; w < kMW; ++w) {
            a.x += lds.sum[w][lane][2 * c];
            a.y += lds.sum[w][lane][2 * c + 1];
        }
        part[((long long)blockIdx.y * nc + c0 + c) * M + sh * shot_len + o] = a;
    }
}

template <int CT, bool R2>
__global__ void __launch_bounds__(64 * kMW) k_gdft_adj_mfma(
    const float* __restrict__ kx, const float* __restrict__ ky, const float* __restrict__ kz,
    const float* __restrict__ t, const float* __restrict__ ix, const float* __restrict__ iy,
    const float* __restrict__ iz, const float* __restrict__ fm, const float2* __restrict__ y,
    long long ystride, const float2* __restrict__ S, int nc, int M, int N, int slice_len,
    int shot_len, long long s_shot, float2* __restrict__ part, R2Args r2)
{
    __shared__ MfmaLds<CT> lds;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int o0 = blockIdx.x * 64;
    // gridDim.y / nshot slices per shot, each within its shot
    const int sps = (int)gridDim.y / (M / shot_len);
    const int sh = blockIdx.y / sps;
    const int i0 = sh * shot_len + (blockIdx.y - sh * sps) * slice_len;
    const int i1 = min(sh * shot_len + shot_len, i0 + slice_len);
    if (S) S += sh * s_shot;
    float4 co[4];
    float3 go[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int j = min(o0 + 16 * u + (lane & 15), N - 1);
        co[u] = make_float4(ix[j], iy[j], iz[j], (float)((double)fm[j] / (2.0 * M_PI)));
        go[u] = R2 ? make_float3(r2.gx[j], r2.gy[j], r2.gz[j]) : make_float3(0.f, 0.f, 0.f);
    }
    const int quarter = ((max(i1 - i0, 0) + 4 * kMW - 1) / (4 * kMW)) * 4;
    const int q0 = min(i1, i0 + wv * quarter), q1 = min(i1, q0 + quarter);
    const int o = min(o0 + lane, N - 1);
    double gr = 0.0, gi = 0.0;
    for (int c0 = 0; c0 < nc; c0 += 8 * CT) {
        pgd_f4 acc[4][CT];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[u][c] = pgd_f4{0.f, 0.f, 0.f, 0.f};
        if (c0) __syncthreads();  // the previous coils' sums are read
        dft_products<CT, R2, true>(
            co, go, q0, q1, lds.in.v[wv], lds.in.r[wv], lds.in.g[wv], r2,
            [&](int q, bool ok, float* row, float4& rr, float3&) {
                const int qc = ok ? q : 0;
                rr = make_float4(kx[qc], ky[qc], kz[qc], t[qc]);
                float2 v[8 * CT];
#pragma unroll
                for (int c = 0; c < 8 * CT; ++c) v[c] = y[min(c0 + c, nc - 1) * ystride + qc];
#pragma unroll
                for (int c = 0; c < 8 * CT; ++c) {
                    const bool on = ok && c0 + c < nc;
                    row[2 * c] = on ? v[c].x : 0.f;
                    row[2 * c + 1] = on ? v[c].y : 0.f;
                }
            },
            acc);
        __syncthreads();
        dft_store<CT>(lds.sum[wv], acc);
        __syncthreads();
        // output o, this wavefront's 2 CT coils: conj(S_c) times the sums
#pragma unroll
        for (int u = 0; u < 2 * CT; ++u) {
            const int c = wv * 2 * CT + u;
            if (c0 + c >= nc) break;
            float2 a = make_float2(lds.sum[0][lane][2 * c], lds.sum[0][lane][2 * c + 1]);
#pragma unroll
            for (int w = 1; w < kMW; ++w) {
                a.x += lds.sum[w][lane][2 * c];
                a.y += lds.sum[w][lane][2 * c + 1];
            }
            double vr = a.x, vi = a.y;
            if (S) {
                const float2 s = S[(long long)(c0 + c) * N + o];
                const double tr = vr * s.x + vi * s.y;
                const double ti = vi * s.x - vr * s.y;
                vr = tr;
                vi = ti;
            }
            gr += vr;
            gi += vi;
        }
    }
    // the four wavefronts' coils, in order
    __syncthreads();
    double2* red = reinterpret_cast<double2*>(&lds);
    static_assert(sizeof(lds) >= kMW * 64 * sizeof(double2), "coil sums");
    red[wv * 64 + lane] = make_double2(gr, gi);
    __syncthreads();
    if (wv == 0 && o0 + lane < N) {
        for (int w = 1; w < kMW; ++w) {
            gr += red[w * 64 + lane].x;
            gi += red[w * 64 + lane].y;
        }
        part[(long long)blockIdx.y * N + o] = make_float2((float)gr, (float)gi);
    }
}

// out[(i / row) * ostride + i % row] (+)= sum of the slices of element i:
// each run of `group` consecutive slices is summed in slice order, and the
// runs are added in order
__global__ void k_sum_slices(const float2* part, int nslice, int group, long long n,
                             long long row, long long ostride, int acc, float2* out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float2 s = make_float2(0.f, 0.f);
    for (int g0 = 0; g0 < nslice; g0 += group) {
        float2 t = part[(long long)g0 * n + i];
#pragma unroll 8
        for (int k = g0 + 1; k < g0 + group; ++k) {
            const float2 p = part[(long long)k * n + i];
            t.x += p.x;
            t.y += p.y;
        }
        s = g0 ? make_float2(s.x + t.x, s.y + t.y) : t;
    }
    const long long r = i / row;
    const long long o = r * ostride + (i - r * row);
    if (acc) {
        const float2 a = out[o];
        s = make_float2(a.x + s.x, a.y + s.y);
    }
    out[o] = s;
}

void sum_slices(const float2* part, int nslice, int group, long long n, long long row,
                long long ostride, int acc, float2* out, hipStream_t s)
{
    // (short outputs in blocks of one wavefront, to spread over the chip)
    const int nt = n < 65536 ? 64 : 256;
    hipLaunchKernelGGL(k_sum_slices, dim3((unsigned)((n + nt - 1) / nt)), dim3(nt), 0, s, part,
                       nslice, group, n, row, ostride, acc, out);
}

R2Args r2_args(const pgd::DftData& d)
{
    return R2Args{d.gx, d.gy, d.gz, 1.0f / (float)d.numx, 1.0f / (float)d.numy,
                  1.0f / (float)d.numz};
}

// slices per shot: aim for >= 4096 wavefronts in flight, each slice at
// least 64 inputs (small problems, such as pcSENSE's DFTs of ~1k samples a
// shot, would otherwise leave most of the 1024 SIMDs idle)
int slices_for(long long outputs, long long inputs, int nshot = 1)
{
    long long waves = (outputs + kT - 1) / kT;
    int s = 1;
    while (waves * nshot * s < 4096 && inputs / (s * 2) >= 64 && nshot * s < 64) s *= 2;
    return s;
}

// the matrix-core kernels split a slice over the block's wavefronts, so the
// same wavefronts are in flight with a quarter of the slices
int mfma_slices(int slices) { return slices / kMW > 1 ? slices / kMW : 1; }

}  // namespace

namespace pgd {

size_t part_elems(int M, int N, int nc, bool adjoint, int nshot)
{
    if (adjoint) return (size_t)slices_for(N, M / nshot, nshot) * nshot * N;
    return (size_t)slices_for((long long)M, N) * nc * M;
}

void forward(const DftData& d, const float2* x, const float2* S, int nc, float2* out, float2* part,
             hipStream_t s, long long ostride, int nshot, long long s_shot)
{
    if (ostride < 0) ostride = d.M;
    if (nshot < 1 || d.M % nshot)
        throw pg::Error{PG_ERR_ARG, "the DFT's shots must split its samples evenly"};
    const int shot_len = d.M / nshot;
    const R2Args r2 = r2_args(d);
    int ns;
    if (d.precision == 1) {
        ns = slices_for(d.M, d.N);
        const int slen = (d.N + ns - 1) / ns;
        constexpr int NCB = 8;
        const dim3 grid(nshot * ((shot_len + kT - 1) / kT), ns, (nc + NCB - 1) / NCB);
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(kT), 0, s, d.kx, d.ky, d.kz, d.t, d.ix, d.iy, d.iz,
                               d.fm, x, S, nc, d.M, d.N, slen, shot_len, s_shot, part, r2);
        };
        d.gx ? launch(k_gdft_fwd<NCB, true>) : launch(k_gdft_fwd<NCB, false>);
    } else {
        ns = mfma_slices(slices_for(d.M, d.N));
        const int slen = (d.N + ns - 1) / ns;
        auto launch = [&](auto kern, int coils) {
            hipLaunchKernelGGL(kern, dim3(nshot * ((shot_len + 63) / 64), ns, (nc + coils - 1) / coils),
                               dim3(64 * kMW), 0, s, d.kx, d.ky, d.kz, d.t, d.ix, d.iy, d.iz, d.fm, x,
                               S, nc, d.M, d.N, slen, shot_len, s_shot, part, r2);
        };
        // columns for 8 or (in chunks of) 16 coils
        if (nc <= 8)
            d.gx ? launch(k_gdft_fwd_mfma<1, true>, 8) : launch(k_gdft_fwd_mfma<1, false>, 8);
        else
            d.gx ? launch(k_gdft_fwd_mfma<2, true>, 16) : launch(k_gdft_fwd_mfma<2, false>, 16);
    }
    const long long n = (long long)nc * d.M;
    sum_slices(part, ns, ns, n, (long long)d.M, ostride, 0, out, s);
}

void adjoint(const DftData& d, const float2* y, const float2* S, int nc, float2* out, float2* part,
             hipStream_t s, long long ystride, bool accumulate, int nshot, long long s_shot)
{
    if (ystride < 0) ystride = d.M;
    if (nshot < 1 || d.M % nshot)
        throw pg::Error{PG_ERR_ARG, "the DFT's shots must split its samples evenly"};
    const int shot_len = d.M / nshot;
    const R2Args r2 = r2_args(d);
    int sps = slices_for(d.N, shot_len, nshot);
    if (d.precision != 1) sps = mfma_slices(sps);
    const int slen = (shot_len + sps - 1) / sps;
    if (d.precision == 1) {
        constexpr int NCB = 8;
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3((d.N + kT - 1) / kT, nshot * sps), dim3(kT), 0, s, d.kx,
                               d.ky, d.kz, d.t, d.ix, d.iy, d.iz, d.fm, y, ystride, S, nc, d.M, d.N,
                               slen, shot_len, s_shot, part, r2);
        };
        d.gx ? launch(k_gdft_adj<NCB, true>) : launch(k_gdft_adj<NCB, false>);
    } else {
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3((d.N + 63) / 64, nshot * sps), dim3(64 * kMW), 0, s, d.kx,
                               d.ky, d.kz, d.t, d.ix, d.iy, d.iz, d.fm, y, ystride, S, nc, d.M, d.N,
                               slen, shot_len, s_shot, part, r2);
        };
        if (nc <= 8)
            d.gx ? launch(k_gdft_adj_mfma<1, true>) : launch(k_gdft_adj_mfma<1, false>);
        else
            d.gx ? launch(k_gdft_adj_mfma<2, true>) : launch(k_gdft_adj_mfma<2, false>);
    }
    sum_slices(part, nshot * sps, sps, (long long)d.N, (long long)d.N, (long long)d.N,
               accumulate ? 1 : 0, out, s);
}

size_t static_scratch_elems() { return kScratchElems; }

float2* static_scratch()
{
    constexpr int kMaxDev = 64;
    static std::mutex mu;
    static float2* addr[kMaxDev] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev)
        throw pg::Error{PG_ERR_HIP, "no current device for the static scratch"};
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            throw pg::Error{PG_ERR_HIP, std::string("hipGetSymbolAddress(scratch) failed: ") +
                                            hipGetErrorString(e)};
        addr[dev] = (float2*)p;
    }
    return addr[dev];
}

}  // namespace pgd
