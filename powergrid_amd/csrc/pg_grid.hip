// pg_grid.hip -- Kaiser-Bessel interpolation (forward gather) and spreading
// (adjoint scatter) on the oversampled grid, batched over coils x segments.
//
// Tap weights are precomputed per sample (pg_gnufft.h); taps outside the
// clamped window of gridding.cpp:67-73 carry weight 0 and their addresses
// are clamped into the grid, so no tap wraps around.
//
// interp  -- 2-D, large batches: by 4x4 grid patches on the matrix cores, the
//            samples' shares added in a second pass (k_interp_mm).  2-D with
//            2..16 segments otherwise: the grid region under a tile of
//            samples is staged in LDS for all or four segments of a coil.
//            3-D: the region under an 8^3 tile, a segment at a time
//            (k_interp3_lds).  Else four lanes per (sample, coil) gather from
//            global memory.  In all, the L segment grids of a coil are read
//            with the same weights and summed with the AA weights
//            (TimeSegmentation.cpp:279-295); the staged forms map coils to
//            XCDs so that each XCD's L2 holds its coils' grids.
// spread  -- first the value of every (sample, grid) pair is formed once
//            (AA weight, CG residual), sample-major.
//            2-D: 4x4 grid patches as products on the matrix cores (patch
//            points x coils x segments) over the samples whose window meets
//            the patch (per-entry patch weights are precomputed); heavy
//            patches are split into runs of <= 64 entries whose sums are
//            added in a fixed order.  No atomics, no zero-fill,
//            deterministic.
//            3-D: 4x4x4 patches on the matrix cores (k_spread3), or, for a few
//            grids of a plan of z-class planes, one thread per sample with
//            hardware float atomics into a zeroed grid (the reference's
//            OpenACC spread, gridding.cpp:102-106).
#include <cfloat>
#include <cmath>

#include "pg_gnufft.h"
#include "pg_internal.h"
#include "pg_fftreg.h"

namespace {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return min(max(v, lo), hi); }

// ---------------------------------------------------------------- interp --
// Four lanes per sample: lane q of a sample reads the taps q, q+4, q+8 (as
// many as NT has) along y of every row, so one load instruction covers 16
// samples x 32 contiguous bytes; the four partial sums are combined with two
// lane shuffles.
template <int NT, bool D3>
__global__ void __launch_bounds__(256) k_interp(
    const int* __restrict__ lo, const float* __restrict__ w, int M, int Gx, int Gy, int Gz,
    const float2* __restrict__ grids, long long G, int nc, int L, const float* __restrict__ AA,
    const float* __restrict__ AAi, float2* __restrict__ out, long long out_cstride, int nsb,
    int xcd_map, const int* __restrict__ pl, long long pstride)
{
    int c, sb;
    const int p = blockIdx.x;
    if (xcd_map) {
        // consecutive block ids go to consecutive XCDs: keep every coil on
        // one XCD (nc is a multiple of 8 here)
        const int xcd = p & 7, r = p >> 3;
        const int cl = r / nsb;
        sb = r - cl * nsb;
        c = cl * 8 + xcd;
    } else {
        c = p / nsb;
        sb = p - c * nsb;
    }
    if (c >= nc) return;
    const int q = threadIdx.x & 3;
    const int i = sb * (int)(blockDim.x >> 2) + (int)(threadIdx.x >> 2);
    const bool valid = i < M;
    const int ii = valid ? i : M - 1;
    const int lx = lo[ii], ly = lo[M + ii];
    const int lz = D3 ? lo[2 * M + ii] : 0;
    // lane q takes the y taps q, q + 4, q + 8 (zero weight past NT)
    constexpr int JY = (NT + 3) / 4;
    float wy[JY];
    int oy[JY];
#pragma unroll
    for (int j = 0; j < JY; ++j) {
        const int jj = q + 4 * j;
        wy[j] = (jj < NT) ? w[(long long)(NT + jj) * M + ii] : 0.f;
        oy[j] = clampi(ly + jj, 0, Gy - 1);
    }
    float wx[NT], wz[D3 ? NT : 1];
    int ox[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        wx[j] = w[(long long)j * M + ii];
        ox[j] = clampi(lx + j, 0, Gx - 1) * Gy;
    }
    long long oz[D3 ? NT : 1];
    if (D3) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            wz[j] = w[(long long)(2 * NT + j) * M + ii];
            oz[j] = (long long)clampi(lz + j, 0, Gz - 1) * Gx * Gy;
        }
    } else {
        wz[0] = 1.f;
        oz[0] = 0;
    }
    // z-class planes (2-D gather on the plane of the sample's class)
    const float2* gp = (!D3 && pl) ? grids + (long long)pl[ii] * pstride : grids;
    float tr = 0.f, ti = 0.f;
#pragma unroll 1
    for (int l = 0; l < L; ++l) {
        const float2* g = gp + ((long long)c * L + l) * G;
        float ar = 0.f, ai = 0.f;
#pragma unroll
        for (int jz = 0; jz < (D3 ? NT : 1); ++jz) {
            const float2* gz = g + oz[jz];
#pragma unroll
            for (int jx = 0; jx < NT; ++jx) {
                const float2* row = gz + ox[jx];
                float rr = 0.f, ri = 0.f;
#pragma unroll
                for (int j = 0; j < JY; ++j) {
                    const float2 v = row[oy[j]];
                    rr += wy[j] * v.x;
                    ri += wy[j] * v.y;
                }
                const float wxz = D3 ? wx[jx] * wz[jz] : wx[jx];
                ar += wxz * rr;
                ai += wxz * ri;
            }
        }
        if (AA) {
            const float a = AA[(long long)l * M + ii];
            if (AAi) {
                // complex weights, real and imaginary parts apart
                const float b = AAi[(long long)l * M + ii];
                const float nr = a * ar - b * ai;
                ai = a * ai + b * ar;
                ar = nr;
            } else {
                ar *= a;
                ai *= a;
            }
        }
        tr += ar;
        ti += ai;
    }
    tr += __shfl_xor(tr, 1);
    ti += __shfl_xor(ti, 1);
    tr += __shfl_xor(tr, 2);
    ti += __shfl_xor(ti, 2);
    if (q == 0 && valid) out[c * out_cstride + i] = make_float2(tr, ti);
}

// ------------------------------------------------- 2-D interp through LDS --
// Sum over the 8 lanes of each aligned 8-lane group with DPP; the total ends
// in the group's lane 7 (row_half_mirror pairs lane k with lane 7 - k).
__device__ __forceinline__ float group8_sum_to_7(float v)
{
#define PG_DPP_ADD8(v, CTRL)                                                                 \
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), (CTRL), 0xF, 0xF, \
                                                    false))
    PG_DPP_ADD8(v, 0xB1);   // quad_perm [1,0,3,2]
    PG_DPP_ADD8(v, 0x4E);   // quad_perm [2,3,0,1]
    PG_DPP_ADD8(v, 0x141);  // row_half_mirror
#undef PG_DPP_ADD8
    return v;
}

// One block per (work item, coil): the kIR x kIR grid region under the
// item's tile is staged in LDS for all L segments of the coil ([x][l][y],
// y fastest, LP segment slots), together with the item's sample records and
// their AA weights.  Each wavefront then takes 8 samples at a time with
// lane = (sample s, segment l):
//   acc_l = sum_x wx[x] sum_y wy[y] g_l(ox + x, oy + y),  value = sum_l AA_l acc_l
// the segment sum being a 3-step DPP reduction inside each 8-lane group.
// Blocks are ordered coil-fastest so that coil c stays on XCD c % 8.
constexpr int kInterpWaves = 8;

template <int LP, bool CPX>
__global__ void __launch_bounds__(64 * kInterpWaves) k_interp_lds(
    const int4* __restrict__ items, const float4* __restrict__ rec, int ity, int padl,
    const float2* __restrict__ grids, long long G, int Gx, int Gy, int nc, int L,
    const float* __restrict__ AA, const float* __restrict__ AAi, int M, float2* __restrict__ out,
    long long out_cstride, long long pstride)
{
    constexpr int R = pg::kIR;
    constexpr int CH = pg::kIChunk;
    __shared__ float2 tile[R * LP * R];
    __shared__ float4 srec[CH * 5];
    __shared__ float saa[CH * LP];
    __shared__ float saai[CPX ? CH * LP : 1];
    const int c = blockIdx.x % nc;
    const int4 it = items[blockIdx.x / nc];
    const int n = it.z - it.y;  // 1..CH
    const int tx = it.x / ity, ty = it.x - (it.x / ity) * ity;
    const int rx0 = tx * pg::kIT - padl, ry0 = ty * pg::kIT - padl;
    // item plane it.w (z-class planes; 0 for a 2-D plan)
    const float2* gc = grids + (long long)it.w * pstride + (long long)c * L * G;
    // Staging: every global load of the block is issued before any LDS
    // store, then one barrier.  The region goes as rows (xr, l) of R values
    // along y, 32 lanes per row (R <= 32), row and segment by shifts, the
    // grid offset in 32 bits (L*G of one coil); only points inside the grid
    // are loaded.  The weights are read with the sample indices taken from
    // the records in global memory.
    static_assert(R <= 32 && (LP & (LP - 1)) == 0, "staging layout");
    constexpr int NTH = 64 * kInterpWaves;
    constexpr int PASS = NTH / 32;                  // rows per pass
    constexpr int NP = (R * LP + PASS - 1) / PASS;  // passes over the rows
    constexpr int NR = (CH * 5 + NTH - 1) / NTH;    // record loads per thread
    constexpr int NA = (CH * LP + NTH - 1) / NTH;   // weight loads per thread
    const int yr = threadIdx.x & 31;
    const int y = ry0 + yr;
    const bool yok = yr < R && y >= 0 && y < Gy;
    // loads from clamped, in-range addresses with the condition applied as a
    // select, so that none of them sits behind a branch and all are in flight
    // together
    const int yc = min(max(y, 0), Gy - 1);
    float2 tv[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const int row = (int)(threadIdx.x >> 5) + k * PASS;
        const int l = row & (LP - 1), xr = row / LP;
        const int x = rx0 + xr;
        const bool ok = row < R * LP && yok && l < L && x >= 0 && x < Gx;
        const int lc = min(l, L - 1), xc = min(max(x, 0), Gx - 1);
        const float2 v = gc[lc * (int)G + xc * Gy + yc];
        tv[k] = ok ? v : make_float2(0.f, 0.f);
    }
    float4 rv[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const int e = min((int)threadIdx.x + k * NTH, n * 5 - 1);
        rv[k] = rec[(long long)it.y * 5 + e];
    }
    float av[NA], aiv[CPX ? NA : 1];
#pragma unroll
    for (int k = 0; k < NA; ++k) {
        const int e = (int)threadIdx.x + k * NTH;
        const int sl = min(e / LP, n - 1), l = e & (LP - 1);
        const bool ok = e < n * LP && l < L;
        const int i = __float_as_int(rec[((long long)it.y + sl) * 5].x);
        const long long o = (long long)min(l, L - 1) * M + i;
        av[k] = ok ? AA[o] : 0.f;
        if (CPX) aiv[k] = ok ? AAi[o] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const int row = (int)(threadIdx.x >> 5) + k * PASS;
        if (row < R * LP && yr < R) tile[row * R + yr] = tv[k];
    }
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const int e = (int)threadIdx.x + k * NTH;
        if (e < n * 5) srec[e] = rv[k];
    }
#pragma unroll
    for (int k = 0; k < NA; ++k) {
        const int e = (int)threadIdx.x + k * NTH;
        if (e < n * LP) {
            saa[e] = av[k];
            if (CPX) saai[e] = aiv[k];
        }
    }
    __syncthreads();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // scalar sample loop
    const int lane = threadIdx.x & 63;
    const int s8 = lane >> 3, l8 = lane & 7;
    for (int base = wv * 8; base < n; base += kInterpWaves * 8) {
        const int sl = min(base + s8, n - 1);
        const float4* rp = srec + sl * 5;
        const float4 h = rp[0];
        const int ox = __float_as_int(h.y), oy = __float_as_int(h.z);
        const float4 xa = rp[1], xb = rp[2], ya = rp[3], yb = rp[4];
        const float wx[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
        const float wy[8] = {ya.x, ya.y, ya.z, ya.w, yb.x, yb.y, yb.z, yb.w};
        float tr = 0.f, ti = 0.f;
#pragma unroll
        for (int g = 0; g < LP / 8; ++g) {
            const int l = g * 8 + l8;
            const float2* tp = tile + ((ox * LP + l) * R + oy);
            float ar = 0.f, ai = 0.f;
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                const float2* row = tp + x * LP * R;
                float rr = 0.f, ri = 0.f;
#pragma unroll
                for (int y = 0; y < 8; ++y) {
                    const float2 v = row[y];
                    rr += wy[y] * v.x;
                    ri += wy[y] * v.y;
                }
                ar += wx[x] * rr;
                ai += wx[x] * ri;
            }
            const float a = saa[sl * LP + l];
            if (CPX) {
                const float b = saai[sl * LP + l];
                tr += a * ar - b * ai;
                ti += a * ai + b * ar;
            } else {
                tr += a * ar;
                ti += a * ai;
            }
        }
        tr = group8_sum_to_7(tr);
        ti = group8_sum_to_7(ti);
        if (l8 == 7 && base + s8 < n)
            out[c * out_cstride + __float_as_int(h.x)] = make_float2(tr, ti);
    }
}

// The same interpolation with the segments staged four at a time: one block
// of 256 threads per (work item of <= 64 samples, coil); lane task = (sample
// s, segment slot l4) with s = tid / 4, so a block's 256 tasks cover its
// item's samples once per chunk of four segments.  Per chunk the 23 x 23
// region of the four segment grids is staged in LDS as [x][y][l] (17 KB: a
// point's four segments side by side, so a sample's four lanes read 32
// contiguous bytes at every tap): a thread loads its points (rows of 23
// along y across the threads: coalesced) from each of the four grids and
// stores each point as two 16-byte writes.  The stores follow the previous
// chunk's taps, and the loads of the next chunk are issued before this
// chunk's taps.  Each task forms
//   acc_l = sum_x wx[x] sum_y wy[y] g_l(ox + x, oy + y)
// and adds AA_l acc_l to its running sum; the four slots of a sample are
// added with two DPP steps at the end.  The sample records go straight to
// registers; the small LDS footprint (21 KB: the region and the AA weights)
// lets seven blocks share a CU, so one block's staging overlaps the others'
// taps.
constexpr int kI4Threads = 256;
constexpr int kI4Chunk = 64;
// the last word of a raw (stride 0) buffer resource on gfx950: 32-bit data
// format, no swizzle; loads at offsets at or past the resource's size return
// zero
constexpr int kBufferWord3 = 0x00020000;

template <bool CPX>
__global__ void __launch_bounds__(kI4Threads, CPX ? 6 : 7) k_interp_lds4(
    const int4* __restrict__ items, const float4* __restrict__ rec, int ity, int padl,
    const float2* __restrict__ grids, long long G, int Gx, int Gy, int nc, int L,
    const float* __restrict__ AA, const float* __restrict__ AAi, int M, float2* __restrict__ out,
    long long out_cstride, long long pstride)
{
    constexpr int R = pg::kIR;
    constexpr int LC = 4;
    constexpr int CH = kI4Chunk;
    constexpr int NTH = kI4Threads;
    constexpr int NQ = R * R;                  // points of the region
    constexpr int NP = (NQ + NTH - 1) / NTH;   // points per thread
    constexpr int PMAX = R + pg::kI4Pitches - 1;
    static_assert(CH * LC == NTH, "one task per thread");
    // the region's R rows at the item's pitch P (R .. PMAX points)
    __shared__ __align__(16) float2 tile[R * PMAX * LC];
    constexpr int NA = (CH * 16 + NTH - 1) / NTH;  // weight loads per thread
    __shared__ float saa[CH * 16];
    __shared__ float saai[CPX ? CH * 16 : 1];
    const int tid = threadIdx.x;
    // blocks (item, coil), coil fastest: the items of coil c run on XCD
    // c % 8, whose L2 serves neighbouring tiles' overlapping regions (item
    // fastest measured 40% slower)
    const int c = blockIdx.x % nc;
    const int4 it = items[blockIdx.x / nc];
    const int n = it.z - it.y;  // 1..CH
    const int tcode = it.x & 0xFFFFFF, P = R + (it.x >> 24);
    const int tx = tcode / ity, ty = tcode - (tcode / ity) * ity;
    const int rx0 = tx * pg::kIT - padl, ry0 = ty * pg::kIT - padl;
    // item plane it.w (z-class planes; 0 for a 2-D plan)
    const float2* gc = grids + (long long)it.w * pstride + (long long)c * L * G;
    const int s = tid >> 2, l4 = tid & 3;
    const bool live = s < n;
    int ox = 0, oy = 0, idx = 0;
    float wx[8], wy[8];
    float tr = 0.f, ti = 0.f;
    // Staging: point q = tid + k NTH of the region (xr = q / R, yr = q % R)
    // sits at byte offset voff[k] in each segment grid, the same for every
    // chunk.  The loads go through one buffer resource per segment slot of
    // the chunk, sized zero for a slot past L: a point outside the x-y grid
    // gets an offset of 2^31, and the hardware returns zero for it and for
    // every load of an empty slot, so the loads need neither clamps nor
    // selects and are all issued back to back.
    int voff[NP], soff[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const int q = tid + k * NTH;
        const int xr = q / R, yr = q - (q / R) * R;
        const int x = rx0 + xr, y = ry0 + yr;
        const bool ok = q < NQ && x >= 0 && x < Gx && y >= 0 && y < Gy;
        voff[k] = ok ? (x * Gy + y) * 8 : (int)0x80000000u;
        soff[k] = (xr * P + yr) * LC;
    }
    float2 tv[NP][LC];
    auto load_chunk = [&](int g) {
#pragma unroll
        for (int lc = 0; lc < LC; ++lc) {
            const bool has = g * LC + lc < L;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(gc + (has ? (long long)(g * LC + lc) * G : 0LL)), (short)0,
                has ? (int)G * 8 : 0, kBufferWord3);
#pragma unroll
            for (int k = 0; k < NP; ++k)
                tv[k][lc] = __builtin_bit_cast(
                    float2, __builtin_amdgcn_raw_buffer_load_b64(rs, voff[k], 0, 0));
        }
    };
    // The task's sample record (into registers: the four lanes of a sample
    // read the same 80 bytes), the sample indices of the (sample, segment
    // slot) pairs e = s * 16 + l, chunk 0 of the region and then the AA
    // weights (by those indices) are all requested before the first LDS
    // store; a record or weight of a sample past n or a slot past L reads
    // zero (offset past the resource's size, or 2^31).
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(rec + (long long)it.y * 5), (short)0, n * 5 * 16, kBufferWord3);
    float4 rv[5];
#pragma unroll
    for (int k = 0; k < 5; ++k)
        rv[k] = __builtin_bit_cast(
            float4, __builtin_amdgcn_raw_buffer_load_b128(rr, (s * 5 + k) * 16, 0, 0));
    int iv[NA];
#pragma unroll
    for (int k = 0; k < NA; ++k) {
        const int e = tid + k * NTH;
        iv[k] = __float_as_int(rec[((long long)it.y + min(e >> 4, n - 1)) * 5].x);
    }
    load_chunk(0);
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)AA, (short)0, L * M * 4, kBufferWord3);
    const __amdgpu_buffer_rsrc_t rai =
        __builtin_amdgcn_make_buffer_rsrc((void*)(CPX ? AAi : AA), (short)0, L * M * 4,
                                          kBufferWord3);
    float av[NA], aiv[CPX ? NA : 1];
#pragma unroll
    for (int k = 0; k < NA; ++k) {
        const int e = tid + k * NTH, l = e & 15;
        const int o = (e >> 4) < n && l < L ? (l * M + iv[k]) * 4 : (int)0x80000000u;
        av[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, o, 0, 0));
        if (CPX)
            aiv[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rai, o, 0, 0));
    }
    auto store_chunk = [&]() {
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            const int q = tid + k * NTH;
            if (q < NQ) {
                float4* t4 = reinterpret_cast<float4*>(tile + soff[k]);
                t4[0] = make_float4(tv[k][0].x, tv[k][0].y, tv[k][1].x, tv[k][1].y);
                t4[1] = make_float4(tv[k][2].x, tv[k][2].y, tv[k][3].x, tv[k][3].y);
            }
        }
    };
    store_chunk();
#pragma unroll
    for (int k = 0; k < NA; ++k) {
        saa[tid + k * NTH] = av[k];
        if (CPX) saai[tid + k * NTH] = aiv[k];
    }
    auto take_record = [&]() {
        const float4 h = rv[0];
        idx = __float_as_int(h.x);
        ox = __float_as_int(h.y);
        oy = __float_as_int(h.z);
        const float4 xa = rv[1], xb = rv[2], ya = rv[3], yb = rv[4];
        wx[0] = xa.x; wx[1] = xa.y; wx[2] = xa.z; wx[3] = xa.w;
        wx[4] = xb.x; wx[5] = xb.y; wx[6] = xb.z; wx[7] = xb.w;
        wy[0] = ya.x; wy[1] = ya.y; wy[2] = ya.z; wy[3] = ya.w;
        wy[4] = yb.x; wy[5] = yb.y; wy[6] = yb.z; wy[7] = yb.w;
    };
    // the taps of chunk g (in LDS) for this task's segment
    auto taps = [&](int g) {
        const int l = g * LC + l4;
        if (live && l < L) {
            const float2* tp = tile + ((ox * P + oy) * LC + l4);
            float ar = 0.f, ai = 0.f;
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                const float2* row = tp + x * P * LC;
                float rr = 0.f, ri = 0.f;
#pragma unroll
                for (int y = 0; y < 8; ++y) {
                    const float2 v = row[y * LC];
                    rr += wy[y] * v.x;
                    ri += wy[y] * v.y;
                }
                ar += wx[x] * rr;
                ai += wx[x] * ri;
            }
            const float a = saa[s * 16 + l];
            if (CPX) {
                const float b = saai[s * 16 + l];
                tr += a * ar - b * ai;
                ti += a * ai + b * ar;
            } else {
                tr += a * ar;
                ti += a * ai;
            }
        }
    };
    for (int g = 0;; ++g) {
        __syncthreads();  // chunk g is in LDS
        if (g == 0) take_record();
        // the next chunk's loads are in flight during this chunk's taps
        const bool more = (g + 1) * LC < L;
        if (more) load_chunk(g + 1);
        taps(g);
        if (!more) break;
        __syncthreads();  // chunk g's taps are done
        store_chunk();
    }
    // the four segment slots of a sample (a quad of lanes)
#define PG_DPP_ADDQ(v, CTRL)                                                                 \
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), (CTRL), 0xF, 0xF, \
                                                    false))
    PG_DPP_ADDQ(tr, 0xB1);  // quad_perm [1,0,3,2]
    PG_DPP_ADDQ(ti, 0xB1);
    PG_DPP_ADDQ(tr, 0x4E);  // quad_perm [2,3,0,1]
    PG_DPP_ADDQ(ti, 0x4E);
#undef PG_DPP_ADDQ
    if (l4 == 0 && live) out[c * out_cstride + idx] = make_float2(tr, ti);
}

// The full 3-D grid with 6 or 8 taps: one block of 512 threads per (work item
// of <= kI3Chunk samples whose window starts lie in one 8^3 tile, coil).
// Per segment the R^3 region under the tile (R = 7 + NT) is staged in LDS
// through a buffer resource (points outside the grid read zero), the next
// segment's loads in flight during the taps.  Thread (s, y) = (tid / 8,
// tid % 8) sums sample s over the x and z taps at y tap y:
//   t = sum_z wz sum_x wx g(ox + x, oy + y, oz + z),
// adds AA_l t to its running sum, and the 8 lanes of a sample are added at
// the end with their wy.  A half-wavefront's tap read is then 4 runs of 64
// bytes (32 separate samples would collide 3.5-fold on the banks, 4 runs
// about twofold).  Each XCD takes one run of the items (in Morton order of
// their tiles), one coil after another: the regions of a coil's L grids under
// some sixteen neighbouring tiles then fit its L2.
// Measured on 32 grids of 128^3, 131072 samples on 1024 spokes: 2130 us for
// the gather kernel above (four lanes per sample: 16 cache lines per load),
// 1830 us for a wavefront per sample gathering 8 rows of 64 bytes per load,
// 690 us here.  Bound by the LDS, busy for 71% of the time (27% in bank
// conflicts), beside the vector units' 41%.
using pg::kI3Chunk;

template <int NT, bool CPX>
__global__ void __launch_bounds__(8 * kI3Chunk) k_interp3_lds(
    const int4* __restrict__ items, int n_items, const int4* __restrict__ rec,
    const float* __restrict__ wpad, int itx, int ity, int padl, const float2* __restrict__ grids,
    long long G, int Gx, int Gy, int Gz, int nc, int L, const float* __restrict__ AA,
    const float* __restrict__ AAi, int M, float2* __restrict__ out, long long out_cstride, int per)
{
    constexpr int R = 7 + NT;
    constexpr int NQ = R * R * R;
    constexpr int NTH = 8 * kI3Chunk;
    constexpr int NP = (NQ + NTH - 1) / NTH;
    constexpr int NTP = 16;
    __shared__ float2 tile[NQ];
    const int tid = threadIdx.x;
    const int p = blockIdx.x, pr = p >> 3;
    const int c = pr / per, k = (p & 7) * per + pr - c * per;
    if (k >= n_items) return;
    const int4 it = items[k];
    const int n = it.z - it.y;
    const int tx = it.x % itx, tr0 = it.x / itx;
    const int rx0 = tx * 8 - padl, ry0 = (tr0 % ity) * 8 - padl, rz0 = (tr0 / ity) * 8 - padl;
    const float2* gc = grids + (long long)c * L * G;
    int voff[NP];
#pragma unroll
    for (int u = 0; u < NP; ++u) {
        const int q = tid + u * NTH;
        const int zr = q / (R * R), w = q - zr * (R * R);
        const int xr = w / R, yr = w - xr * R;
        const int x = rx0 + xr, y = ry0 + yr, z = rz0 + zr;
        const bool ok = q < NQ && x >= 0 && x < Gx && y >= 0 && y < Gy && z >= 0 && z < Gz;
        voff[u] = ok ? ((z * Gx + x) * Gy + y) * 8 : (int)0x80000000u;
    }
    float2 tv[NP];
    auto load_segment = [&](int l) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(gc + l * G), (short)0, (int)G * 8, kBufferWord3);
#pragma unroll
        for (int u = 0; u < NP; ++u)
            tv[u] = __builtin_bit_cast(float2,
                                       __builtin_amdgcn_raw_buffer_load_b64(rs, voff[u], 0, 0));
    };
    load_segment(0);
    const int s = tid >> 3, ty = tid & 7;
    const bool live = s < n && ty < NT;
    const int4 r = rec[it.y + min(s, n - 1)];
    const int ox = r.y & 255, oy = (r.y >> 8) & 255, oz = r.y >> 16;
    const float2* tp = tile + (oz * R + ox) * R + oy + ty;
    // the weights from the re-based window start on (taps moved off it carry
    // weight zero)
    const float* wp = wpad + (long long)r.x * (3 * NTP) + 3;
    const int sx = r.z & 255, sy = (r.z >> 8) & 255, sz = r.z >> 16;
    float wx[NT], wz[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        wx[q] = q + sx < NT ? wp[q + sx] : 0.f;
        wz[q] = q + sz < NT ? wp[2 * NTP + q + sz] : 0.f;
    }
    const float wy = ty + sy < NT ? wp[NTP + ty + sy] : 0.f;
    float tr = 0.f, ti = 0.f;
#pragma unroll 1
    for (int l = 0; l < L; ++l) {
        if (l) __syncthreads();  // the previous segment's taps are done
#pragma unroll
        for (int u = 0; u < NP; ++u)
            if (u + 1 < NP || tid + u * NTH < NQ) tile[tid + u * NTH] = tv[u];
        __syncthreads();
        if (l + 1 < L) load_segment(l + 1);
        if (live) {
            const float a = AA ? AA[(long long)l * M + r.x] : 1.f;
            const float b = CPX ? AAi[(long long)l * M + r.x] : 0.f;
            float ar = 0.f, ai = 0.f;
#pragma unroll
            for (int z = 0; z < NT; ++z) {
                float xr = 0.f, xi = 0.f;
#pragma unroll
                for (int x = 0; x < NT; ++x) {
                    const float2 v = tp[(z * R + x) * R];
                    xr += wx[x] * v.x;
                    xi += wx[x] * v.y;
                }
                ar += wz[z] * xr;
                ai += wz[z] * xi;
            }
            if (CPX) {
                tr += a * ar - b * ai;
                ti += a * ai + b * ar;
            } else {
                tr += a * ar;
                ti += a * ai;
            }
        }
    }
    const float vr = group8_sum_to_7(live ? wy * tr : 0.f);
    const float vi = group8_sum_to_7(live ? wy * ti : 0.f);
    if (ty == 7 && s < n) out[c * out_cstride + r.x] = make_float2(vr, vi);
}

// value of sample i in grid b: AA_l * (in_c[i] or W (y_c[i] - Ax_c[i])),
// the residual formed in FP64 from the FP64 Ax of the CG
__device__ __forceinline__ float2 spread_value(const float2* __restrict__ in, long long in_cstride,
                                               const float2* __restrict__ resid_y,
                                               const double2* __restrict__ ax64,
                                               const float* __restrict__ Wd,
                                               const float* __restrict__ AA,
                                               const float* __restrict__ AAi, int L, int M, int b,
                                               int i)
{
    const int c = b / L, l = b - c * L;
    const long long di = c * in_cstride + i;
    float2 v;
    if (resid_y) {
        // W % (yi - Ax)   (solve_pwls_pcg.hpp:83)
        const float2 yv = resid_y[di];
        const double2 a = ax64[di];
        double rr = (double)yv.x - a.x, ri = (double)yv.y - a.y;
        if (Wd) {
            const double wv = Wd[di];
            rr *= wv;
            ri *= wv;
        }
        v = make_float2((float)rr, (float)ri);
    } else {
        v = in[di];
    }
    if (AA) {
        // conj(AA) % d  (TimeSegmentation.cpp:304-310); AAi, when set, holds
        // the imaginary parts of complex weights
        const float a = AA[(long long)l * M + i];
        if (AAi) {
            const float b = AAi[(long long)l * M + i];
            v = make_float2(a * v.x + b * v.y, a * v.y - b * v.x);
        } else {
            v = make_float2(a * v.x, a * v.y);
        }
    }
    return v;
}

// V[i*B + b] = value of sample i in grid b, formed once per spread so that the
// spread kernels read one contiguous row of B values per sample.  Block:
// 4 samples x 64 lanes over b.  (Inside the PCG the update kernel forms the
// next iteration's values itself, with the same arithmetic.)
__global__ void __launch_bounds__(256) k_spread_values(
    const float2* __restrict__ in, long long in_cstride, const float2* __restrict__ resid_y,
    const double2* __restrict__ ax64, const float* __restrict__ Wd, int L,
    const float* __restrict__ AA, const float* __restrict__ AAi, int M, int B,
    float2* __restrict__ V)
{
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= M) return;
    for (int b = threadIdx.x & 63; b < B; b += 64)
        V[(long long)i * B + b] =
            spread_value(in, in_cstride, resid_y, ax64, Wd, AA, AAi, L, M, b, i);
}

// the same for an even grid count, two grids per thread (16-byte stores;
// consecutive threads fill consecutive pairs of a sample's row)
__global__ void __launch_bounds__(256) k_spread_values2(
    const float2* __restrict__ in, long long in_cstride, const float2* __restrict__ resid_y,
    const double2* __restrict__ ax64, const float* __restrict__ Wd, int L,
    const float* __restrict__ AA, const float* __restrict__ AAi, int M, int B,
    float2* __restrict__ V)
{
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int hb = B >> 1;
    const long long i = p / hb;
    if (i >= M) return;
    const int b = 2 * (int)(p - i * hb);
    const float2 v0 = spread_value(in, in_cstride, resid_y, ax64, Wd, AA, AAi, L, M, b, (int)i);
    const float2 v1 = spread_value(in, in_cstride, resid_y, ax64, Wd, AA, AAi, L, M, b + 1, (int)i);
    *reinterpret_cast<float4*>(V + i * B + b) = make_float4(v0.x, v0.y, v1.x, v1.y);
}

void launch_values(const float2* in, long long in_cstride, const float2* resid_y,
                   const double2* ax64, const float* Wd, int L, const float* AA, const float* AAi,
                   int M, int B, float2* V, hipStream_t s)
{
    if (B % 2 == 0) {
        const long long n = (long long)M * (B / 2);
        hipLaunchKernelGGL(k_spread_values2, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, in,
                           in_cstride, resid_y, ax64, Wd, L, AA, AAi, M, B, V);
    } else {
        hipLaunchKernelGGL(k_spread_values, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, s, in,
                           in_cstride, resid_y, ax64, Wd, L, AA, AAi, M, B, V);
    }
}

// Compact sample rows for the spread of a time-segmented batch: row i holds
// the nc coil values r_c(i) (the input, or W (y - Ax) rounded to FP32, as
// spread_value forms them) as float2, then the L segment weights AA_l(i) (and,
// for complex weights, their imaginary parts), padded to S floats (a multiple
// of 4).  The spread forms each grid's value AA_l r_c from the row, with the
// products of spread_value, so both spreads sum the same values; the rows
// are S floats per sample instead of 2 nc L.  Block: 64 samples, staged in
// LDS and written out as contiguous rows.
__global__ void __launch_bounds__(256) k_spread_rows(
    const float2* __restrict__ in, long long in_cstride, const float2* __restrict__ resid_y,
    const double2* __restrict__ ax64, const float* __restrict__ Wd, int L,
    const float* __restrict__ AA, const float* __restrict__ AAi, int M, int nc, int S,
    float* __restrict__ rows)
{
    extern __shared__ float buf[];  // 64 x S
    const int i0 = blockIdx.x * 64;
    const int tid = threadIdx.x;
    const int n = min(64, M - i0);
    for (int e = tid; e < nc * 64; e += 256) {
        const int c = e >> 6, k = e & 63;
        float2 v = make_float2(0.f, 0.f);
        if (k < n) v = spread_value(in, in_cstride, resid_y, ax64, Wd, nullptr, nullptr, 1, M, c,
                                    i0 + k);
        buf[k * S + 2 * c] = v.x;
        buf[k * S + 2 * c + 1] = v.y;
    }
    const int na = AAi ? 2 * L : L;
    for (int e = tid; e < na * 64; e += 256) {
        const int q = e >> 6, k = e & 63;
        const int i = min(i0 + k, M - 1);
        buf[k * S + 2 * nc + q] = q < L ? AA[(long long)q * M + i] : AAi[(long long)(q - L) * M + i];
    }
    for (int e = tid; e < (S - 2 * nc - na) * 64; e += 256) {
        const int q = e >> 6, k = e & 63;
        buf[k * S + 2 * nc + na + q] = 0.f;
    }
    __syncthreads();
    float* dst = rows + (long long)i0 * S;
    for (int e = tid; e < n * S; e += 256) dst[e] = buf[e];
}

void launch_rows(const float2* in, long long in_cstride, const float2* resid_y, const double2* ax64,
                 const float* Wd, int L, const float* AA, const float* AAi, int M, int nc, int S,
                 float2* rows, hipStream_t s)
{
    hipLaunchKernelGGL(k_spread_rows, dim3((unsigned)((M + 63) / 64)), dim3(256),
                       sizeof(float) * 64 * S, s, in, in_cstride, resid_y, ax64, Wd, L, AA, AAi, M,
                       nc, S, reinterpret_cast<float*>(rows));
}

// ------------------------------------------------- 2-D patch spread --------
// A block of W = kSpreadWaves wavefronts; wavefront w runs the work item
// witems[W block + w] = {patch (-1: none), entry begin, entry end, slot} of at
// most 64 entries for one chunk of the grids: a 4x4 patch as products on the
// matrix cores,
//   acc_l[16 points][16 CT floats] += W[16 points][4 entries] (AA_l r)[4 entries][16 CT floats]
// four entries a step, v_mfma_f32_16x16x4f32 (A[i][k] in lane i + 16k, B[k][j]
// in lane j + 16k, D[i][j] in lane j + 16 (i / 4), register i % 4).  W are the
// entries' 16 weights wx wy (ew, precomputed in FP64: a step's 64 are
// contiguous), r the coil values of up to 8 CT coils in the entry's sample row
// (re and im as separate columns, lane j holding floats CT j .. CT j + CT - 1)
// and AA_l its weights of up to NL segments, so a chunk is NL segments of 8 CT
// coils; the rows are those of k_spread_rows (stride S: nc coil values, then
// L weights, and for MODE 2 their L imaginary parts: conj(AA) r).  MODE 0: no
// weights, the rows hold the nc = B grid values themselves (L = 1).
// A patch of 65 .. 64 W entries is split over gs = 2 .. W consecutive
// wavefronts of a block (bgs[block] = gs, the same for all groups of a block),
// whose sums are added through LDS in a fixed tree order; the group's first
// wavefront writes the patch, or its partial slot when the patch is one of the
// parts of a heavier patch (added by k_spread_heavy_combine).  No atomics, no
// zero-fill, deterministic.
//
// Why this form.  With a lane per grid and the 16 sums of a patch in registers
// (the rows staged in LDS) an entry took 32 FMAs and some 18 more vector
// instructions per 64 grids, 200 clocks, and five LDS broadcasts; here it takes
// 64 clocks of the matrix cores and some 60 of the vector units.  The patches
// of a strip of 16 points along y belong to one block and leave the L2 as
// whole lines (in any order of patches 32-byte pieces reach 0.75 TB/s: 8.6 ms
// for the 6.4 GB of the planes below), and the chunks of a block follow each
// other on one XCD, whose L2 then holds their shared rows and weights (6.0 ->
// 0.55 GB read).  Measured: 384 grids on 32 planes of 256^2, 524288 samples
// (32 coils, 12 segments): 4.92 ms -> 3.03 with the lane per grid in these
// orders -> 2.45 (6.9 GB, 2.8 TB/s; matrix cores 34% busy, vector units 36%);
// 64 grids of 256^2, 32768 samples (8 coils, 8 segments): 30.6 -> 26 us; 4 grids
// of 128^2, 4096 samples: 13.0 -> 4.7 us.
using pg::kSpreadWaves;
typedef float pg_f4 __attribute__((ext_vector_type(4)));
typedef float pg_f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float pg_f2u __attribute__((ext_vector_type(2), aligned(4)));

// a lane's neighbour in its pair (quad_perm [1,0,3,2])
__device__ __forceinline__ float pair_swap(float v)
{
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}

template <int N>
__device__ __forceinline__ void load_floats(const float* p, float (&v)[N])
{
    if constexpr (N == 1) {
        v[0] = p[0];
    } else if constexpr (N == 2) {
        const pg_f2u q = *reinterpret_cast<const pg_f2u*>(p);
        v[0] = q[0];
        v[1] = q[1];
    } else {
#pragma unroll
        for (int u = 0; u < N / 4; ++u) {
            const pg_f4u q = *reinterpret_cast<const pg_f4u*>(p + 4 * u);
#pragma unroll
            for (int t = 0; t < 4; ++t) v[4 * u + t] = q[t];
        }
    }
}

template <int CT, int NL, int MODE>
__global__ void __launch_bounds__(64 * kSpreadWaves) k_spread2(
    const int4* __restrict__ witems, const int* __restrict__ bgs, const int* __restrict__ entries,
    const float* __restrict__ ew, int npy, const float* __restrict__ rows, int S, int nc, int L,
    int ncc, int nch, float2* __restrict__ grids, long long G, int Gy,
    float2* __restrict__ partial, int B, int npp, long long pstride, int gather)
{
    static_assert(MODE || NL == 1, "value rows have no segments");
    constexpr int NA = 4 * NL * CT;  // floats of the patch per lane
    // the block's strips on their way out: LP segments at a time, per coil 4
    // rows of 16 points (the coils' 128 floats 4 apart, against bank conflicts)
    constexpr int LP = NL * CT > 4 ? 4 / CT : NL;
    constexpr int CP = 132;
    constexpr int NS = kSpreadWaves / 4;  // strips of a block (gs = 1)
    constexpr int POOL = NA * 64 * kSpreadWaves / 2 > NS * LP * 8 * CT * CP
                             ? NA * 64 * kSpreadWaves / 2
                             : NS * LP * 8 * CT * CP;
    __shared__ __align__(16) float pool[POOL];
    float(*red)[NA][64] = reinterpret_cast<float(*)[NA][64]>(pool);
    // wave-uniform (scalar) work item
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // block id: XCD, chunk, block of that XCD (chunks fastest)
    const int pr = blockIdx.x >> 3, chunk = pr % nch;
    const int blk = (pr / nch) * 8 + (blockIdx.x & 7);
    const int4 it = witems[blk * kSpreadWaves + wv];
    const int gs = bgs[blk];
    const int c0 = (chunk % ncc) * 8 * CT, l0 = (chunk / ncc) * NL;
    const int nf = 2 * min(8 * CT, nc - c0), nl = min(NL, L - l0);
    const int i = lane & 15, k = lane >> 4;
    // this lane's floats of a row; past the chunk's its last ones (those
    // columns are never stored), an odd coil's last pair moved into place (CT
    // 4, nf % 4 == 2; a last chunk of one coil reads from the coil before it)
    const int ro = 2 * c0 + min(CT * i, nf - CT);
    const bool shifted = CT == 4 && CT * i + CT > nf && CT * i < nf;
    pg_f4 acc[NL][CT];
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
        for (int t = 0; t < CT; ++t) acc[l][t] = pg_f4{0.f, 0.f, 0.f, 0.f};

    // groups of U steps, the next group's loads in flight during this group's
    // products
    constexpr int U = 2;
    const int n = it.z - it.y;  // <= 64
    float w[2][U], v[2][U][CT], a[2][U][NL], ai[2][U][MODE == 2 ? NL : 1];
    if (n > 0) {
        const int es = entries[it.y + min(lane, n - 1)];
        const float* ewl = ew + 16LL * it.y + lane;
        auto load_group = [&](int s, int q) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // (steps past the end: the last step's weights, the last entry)
                w[q][u] = ewl[64 * min(s + u, (n - 1) >> 2)];
                const int si = __shfl(es, min(4 * (s + u) + k, n - 1), 64);
                const float* row = rows + (long long)si * S;
                load_floats<CT>(row + ro, v[q][u]);
                if (MODE) load_floats<NL>(row + 2 * nc + l0, a[q][u]);
                if constexpr (MODE == 2) load_floats<NL>(row + 2 * nc + L + l0, ai[q][u]);
            }
        };
        auto sum_group = [&](int s, int q) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // entries past the end (the last one again): zero weights, and
                // where a caller may see the grid (MODE 0, few grids) zero
                // values, for a sample that is infinite
                const bool in = 4 * (s + u) + k < n;
                const float wm = in ? w[q][u] : 0.f;
                float vm[CT];
#pragma unroll
                for (int t = 0; t < CT; ++t) {
                    vm[t] = v[q][u][t];
                    if (CT == 4 && t < 2) vm[t] = shifted ? v[q][u][(t + 2) % CT] : vm[t];
                    if (CT == 1 && MODE == 0) vm[t] = in ? vm[t] : 0.f;
                }
                // conj(a + i ai) r: the partner of each float, signed
                float vx[MODE == 2 ? CT : 1];
                if constexpr (MODE == 2) {
#pragma unroll
                    for (int t = 0; t < CT; ++t) {
                        const float o = CT == 1 ? pair_swap(vm[0]) : vm[(t ^ 1) % CT];
                        vx[t] = (CT == 1 ? (i & 1) : (t & 1)) ? -o : o;
                    }
                }
#pragma unroll
                for (int l = 0; l < NL; ++l) {
                    if (NL > 1 && l >= nl) break;
#pragma unroll
                    for (int t = 0; t < CT; ++t) {
                        float b = vm[t];
                        if (MODE == 1) b = a[q][u][l] * b;
                        if constexpr (MODE == 2)
                            b = __builtin_fmaf(a[q][u][l], b, ai[q][u][l] * vx[t]);
                        acc[l][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wm, b, acc[l][t], 0, 0, 0);
                    }
                }
            }
        };
        load_group(0, 0);
        for (int s = 0; 4 * s < n; s += 2 * U) {
            load_group(s + U, 1);
            __builtin_amdgcn_sched_barrier(0);
            sum_group(s, 0);
            load_group(s + 2 * U, 0);
            __builtin_amdgcn_sched_barrier(0);
            sum_group(s + U, 1);
        }
    }
    // groups of gs wavefronts: tree sum, wavefront w + r into w
    for (int r = 1; r < gs; r *= 2) {
        __syncthreads();
        if ((wv & (2 * r - 1)) == r)
#pragma unroll
            for (int q = 0; q < NA; ++q) red[wv >> 1][q][lane] = acc[q / (4 * CT)][q / 4 % CT][q % 4];
        __syncthreads();
        if ((wv & (2 * r - 1)) == 0)
#pragma unroll
            for (int q = 0; q < NA; ++q)
                acc[q / (4 * CT)][q / 4 % CT][q % 4] += red[(wv + r) >> 1][q][lane];
    }
    // lane: points (row k, y = 0 .. 3), floats CT i + t of the chunk's coils
    const bool owner = it.x >= 0 && (wv & (gs - 1)) == 0 && CT * i < nf;
    if (gather && 4 * gs <= kSpreadWaves) {
        // strips: four patches along y, of gs wavefronts each, gathered in LDS
        // and stored as whole 128-byte rows, 8 lanes a row
        const int lgs = gs >> 1;  // log2 gs (1 or 2)
        const int st = wv >> (2 + lgs), pi = wv >> lgs & 3;
        // where this thread's piece of a row lies in a grid, per strip (-1:
        // its patch is not of this block)
        const int y2 = threadIdx.x & 7, row = threadIdx.x >> 3 & 3;
        static_assert(NS <= 2, "two strips to a block");
        long long off[NS];
#pragma unroll
        for (int t = 0; t < NS; ++t) {
            const int at = (4 * t + (y2 >> 1)) << lgs;
            const int pt = at < kSpreadWaves ? witems[blk * kSpreadWaves + at].x : -1;
            const int pln = pt / npp, p0 = pt - pln * npp;
            off[t] = pt < 0 ? -1
                            : pln * pstride + (long long)((p0 / npy) * pg::kPatch + row) * Gy +
                                  (p0 % npy) * pg::kPatch + 2 * (y2 & 1);
        }
        for (int lb = 0; lb < nl; lb += LP) {
            __syncthreads();
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                if (l < lb || l >= lb + LP || l >= nl || !owner) continue;
                float* sp = pool + (st * LP + l - lb) * 8 * CT * CP + k * 32 + 8 * pi;
                if constexpr (CT == 1) {
                    // a pair of lanes holds a coil: the even one takes points
                    // 0 and 1, the odd one 2 and 3
                    const bool odd = i & 1;
                    const pg_f4 o = acc[l][0];
                    const float p0 = pair_swap(odd ? o[0] : o[2]);
                    const float p1 = pair_swap(odd ? o[1] : o[3]);
                    reinterpret_cast<float4*>(sp + (i >> 1) * CP)[i & 1] =
                        odd ? make_float4(p0, o[2], p1, o[3]) : make_float4(o[0], p0, o[1], p1);
                } else {
#pragma unroll
                    for (int h = 0; h < CT / 2; ++h) {
                        const pg_f4 re = acc[l][(2 * h) % CT], im = acc[l][(2 * h + 1) % CT];
                        float4* g4 = reinterpret_cast<float4*>(sp + ((CT / 2) * i + h) * CP);
                        g4[0] = make_float4(re[0], im[0], re[1], im[1]);
                        g4[1] = make_float4(re[2], im[2], re[3], im[3]);
                    }
                }
            }
            __syncthreads();
            // pieces of 16 bytes: 8 to a row, 4 rows to a coil (thread % 32);
            // the coils, LP segments and the block's strips in turn
            constexpr int NC = 8 * CT, NQ = NS * LP * NC, QS = 2 * kSpreadWaves;
#pragma unroll
            for (int q0 = 0; q0 < NQ; q0 += QS) {
                const int q = q0 + (int)(threadIdx.x >> 5);
                const int c = q % NC, ll = q / NC % LP, t = q / (NC * LP);
                const long long o = t ? off[NS - 1] : off[0];
                if (q < NQ && t < NS / gs && 2 * c < nf && lb + ll < nl && o >= 0)
                    *reinterpret_cast<float4*>(grids + o +
                                               ((long long)(c0 + c) * L + l0 + lb + ll) * G) =
                        *reinterpret_cast<const float4*>(
                            pool + ((t * LP + ll) * NC + c) * CP + row * 32 + 4 * y2);
            }
        }
        return;
    }
    if (!owner) return;
    const int pln = it.x / npp, q0 = it.x - pln * npp;
    const int px0 = (q0 / npy) * pg::kPatch, py0 = (q0 % npy) * pg::kPatch;
    float2* gp = grids + pln * pstride + (long long)(px0 + k) * Gy + py0;
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        if (l >= nl) break;
        if constexpr (CT == 1) {
            const bool odd = i & 1;
            const pg_f4 o = acc[l][0];
            const float p0 = pair_swap(odd ? o[0] : o[2]), p1 = pair_swap(odd ? o[1] : o[3]);
            const float4 d = odd ? make_float4(p0, o[2], p1, o[3]) : make_float4(o[0], p0, o[1], p1);
            const long long b = (long long)(c0 + (i >> 1)) * L + l0 + l;
            if (it.w >= 0) {
                float2* pp = partial + ((long long)it.w * 16 + 4 * k + 2 * (i & 1)) * B + b;
                pp[0] = make_float2(d.x, d.y);
                pp[B] = make_float2(d.z, d.w);
            } else {
                reinterpret_cast<float4*>(gp + b * G)[i & 1] = d;
            }
        } else {
#pragma unroll
            for (int h = 0; h < CT / 2; ++h) {
                const int c = (CT / 2) * i + h;
                if (2 * c >= nf) break;
                const pg_f4 re = acc[l][(2 * h) % CT], im = acc[l][(2 * h + 1) % CT];
                const long long b = (long long)(c0 + c) * L + l0 + l;
                if (it.w >= 0) {
                    float2* pp = partial + ((long long)it.w * 16 + 4 * k) * B + b;
#pragma unroll
                    for (int r = 0; r < 4; ++r) pp[(long long)r * B] = make_float2(re[r], im[r]);
                } else {
                    float4* g4 = reinterpret_cast<float4*>(gp + b * G);
                    g4[0] = make_float4(re[0], im[0], re[1], im[1]);
                    g4[1] = make_float4(re[2], im[2], re[3], im[3]);
                }
            }
        }
    }
}

// patches summed in parts: add the parts' slots (16 points x B grids) in slot
// order; block (patch, 256 of its 16 B sums)
__global__ void __launch_bounds__(256) k_spread_heavy_combine(
    const int4* __restrict__ comb, int npy, const float2* __restrict__ partial, int B,
    float2* __restrict__ grids, long long G, int Gy, int npp, long long pstride)
{
    const int4 cb = comb[blockIdx.x];
    const int e = blockIdx.y * 256 + threadIdx.x;
    if (e >= 16 * B) return;
    const int q = e / B, b = e - q * B;
    const float2* pp = partial + (long long)cb.y * 16 * B + e;
    float2 t = pp[0];
#pragma unroll 4
    for (int k = 1; k < cb.z; ++k) {
        const float2 v = pp[(long long)k * 16 * B];
        t.x += v.x;
        t.y += v.y;
    }
    const int pln = cb.x / npp, q0 = cb.x - pln * npp;
    const int px0 = (q0 / npy) * pg::kPatch, py0 = (q0 % npy) * pg::kPatch;
    grids[pln * pstride + (long long)b * G + (long long)(px0 + q / pg::kPatch) * Gy + py0 +
          q % pg::kPatch] = t;
}

// the 2-D patches (of every z-class plane) of nc coils x L segments from rows
// of S floats; mode as k_spread2
void launch_spread2(const pg::Gnufft& G, const float* rows, int S, int nc, int L, int mode,
                    float2* grids, long long gsz, long long pstride, float2* partial,
                    hipStream_t s)
{
    const pg::Geometry& g = G.geo;
    const int B = nc * L, npy = g.Gy / pg::kPatch;
    // Whole rows through LDS where the grids outgrow the caches: written as
    // each lane's 16 bytes, a request each, they keep the L2 busy (4e8 of them
    // at the larger size above: 3.36 against 2.45 ms; 64 grids of 128^2 on 16
    // planes, 134 MB: 168 against 161 us for the adjoint); below, the barriers
    // cost more (34 MB: 28.6 against 30.6 us).  Value rows have the shorter loop
    // and gain earlier (16 grids of 512^2, 34 MB, 1000 samples: 55.2 against 51.0
    // us; 64^2 .. 128^2 up to 13 MB: even or 1 us slower).  A single column tile
    // has fewer requests to save while coils are missing: 1 x 8 on 1024^2, 67 MB,
    // 90.8 direct, 98.5 gathered; on 16 planes of 128^2 6 x 8, 101 MB, 128 and 136,
    // 8 x 4, 67 MB, 81 and 85; on 12 planes of 192^2 8 x 4, 113 MB, 128 and 124; on 32
    // planes of 256^2 7 x 4, 470 MB, 503 and 484.
    const double bytes = (G.nzc > 0 && pstride ? G.nzc : 1) * (double)B * gsz * 8;
    const int gather = nc <= 8 ? mode && bytes * nc * nc > 64 * 96e6 : bytes > (mode ? 64e6 : 16e6);
    auto launch = [&](auto kern, int ct, int nseg) {
        const int ncc = (nc + 8 * ct - 1) / (8 * ct), nch = ncc * ((L + nseg - 1) / nseg);
        pg::block_runs(G.n_sblocks, nch, 64 * kSpreadWaves, [&](int o, int n) {
            hipLaunchKernelGGL(kern, dim3((unsigned)n * nch), dim3(64 * kSpreadWaves), 0, s,
                               G.witems + (long long)o * kSpreadWaves, G.bgs + o, G.entries, G.ent_w,
                               npy, rows, S, nc, L, ncc, nch, grids, gsz, g.Gy, partial, B, G.npp,
                               pstride, gather);
        });
    };
    // columns for the coils there are, 8, 16 or chunks of 32, and segments for
    // 16 or 32 sums a lane (8 coils: 4 segments at a time measured 26.2 us,
    // 8 at a time 28.6, at the smaller size above)
    if (mode == 0) {
        if (nc <= 8) launch(k_spread2<1, 1, 0>, 1, 1);
        else if (nc <= 16) launch(k_spread2<2, 1, 0>, 2, 1);
        else launch(k_spread2<4, 1, 0>, 4, 1);
    } else if (mode == 1) {
        if (nc <= 8) launch(k_spread2<1, 4, 1>, 1, 4);
        else if (nc <= 16) launch(k_spread2<2, 4, 1>, 2, 4);
        else launch(k_spread2<4, 2, 1>, 4, 2);
    } else {
        if (nc <= 8) launch(k_spread2<1, 4, 2>, 1, 4);
        else if (nc <= 16) launch(k_spread2<2, 4, 2>, 2, 4);
        else launch(k_spread2<4, 2, 2>, 4, 2);
    }
    if (G.n_comb > 0)
        hipLaunchKernelGGL(k_spread_heavy_combine, dim3(G.n_comb, (16 * B + 255) / 256), dim3(256), 0,
                           s, G.comb, npy, partial, B, grids, gsz, g.Gy, G.npp, pstride);
}

// ------------------------------------------- 2-D interpolation by patches --
// The transpose of k_spread2: the same work items (a patch, at most 64 of its
// entries), for one chunk of 8 CT coils and all L segments:
//   acc[64 entries][16 CT floats] += AA_l (W[entries][16 points] g_l[16 points][16 CT floats])
// over the segments (the weights by FMA: a product's own sum is short, and a
// segment's sum is rounded into acc once), v_mfma_f32_16x16x4f32 with the
// entries as rows: lane (i, k) = (lane % 16, lane / 16) holds entry 16 g + i's
// weights of patch row k (four floats of ew: a group's 1 KB in one load),
// B[k][j] the values of row k of coil j's grid (32 contiguous bytes per lane and
// segment, the next segment's in flight during this one's products).  So every
// grid point is read once, by one block per strip of 128-byte rows; a patch's
// share of each sample goes to part[slot of the entry][coil], the slots of a
// sample in consecutive places, and k_interp_sum adds them in patch order (in
// FP64: an add at the full sum's size for every patch would show in the result).
// Why this form.  The tiled interpolation (k_interp_lds4) reads a tap of 8
// bytes from LDS per FMA pair and is bound by that, by its bank conflicts and
// by the 2.1-fold staged regions; here a value read from memory serves up to 64
// samples, and 64 clocks of the matrix cores take the place of 128 FMAs and 64
// LDS reads per (entry, 64 grids).  Bound by memory requests.  Measured: 384
// grids on 32 planes of 256^2, 524288 samples (32 coils, 12 segments): 3.21 ms ->
// 1.97 + 0.21 for the sums (6.4 GB of grids read and 1.0 of shares written, 3.8
// TB/s; 1.15 GB in the second pass, 5.4 TB/s); 384 grids of 384^2, 65536 samples:
// 380 us -> 214 + 25; 64 grids of 256^2, 32768 samples (8 coils, 8 segments): 35.8
// us -> 27.4 + 5.2.  Slower at the first of these: 32 entries at a time (two
// passes over the values, 2.37 ms), 16 or 8 coils a chunk (2.08, 2.62).
// CT = 1 (up to 8 coils): column j holds the re (j < 8) or im of coil j % 8;
// else tile 2 h holds the re and 2 h + 1 the im of coils 16 h + j.
constexpr int kIpWaves = 4;  // a spread block's items run in blocks of 4 (a strip)
static_assert(kSpreadWaves % kIpWaves == 0, "whole parts of a block");

template <int CT, bool CPLX>
__global__ void __launch_bounds__(64 * kIpWaves) k_interp_mm(
    const int4* __restrict__ witems, const int* __restrict__ entries, const float* __restrict__ ew,
    const int* __restrict__ slots, int npy, const float2* __restrict__ grids, long long G, int Gy,
    int nc, int L, const float* __restrict__ AA, const float* __restrict__ AAi, int M, int ncc,
    float* __restrict__ part, int npp, long long pstride)
{
    constexpr int NH = CT == 1 ? 1 : CT / 2;  // coils per lane
    constexpr int NG = 4;                     // 16-entry groups of an item
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int pr = blockIdx.x >> 3, cc = pr % ncc;
    constexpr int NP = kSpreadWaves / kIpWaves;
    const int blk = pr / ncc / NP * 8 + (blockIdx.x & 7);
    const int4 it = witems[blk * kSpreadWaves + pr / ncc % NP * kIpWaves + wv];
    const int n = it.z - it.y;  // <= 64
    if (it.x < 0 || n <= 0) return;
    const int i = lane & 15, k = lane >> 4;
    const int es = entries[it.y + min(lane, n - 1)], sl = slots[it.y + min(lane, n - 1)];
    const int ng = (n + 15) >> 4;
    float w[NG][4];
#pragma unroll
    for (int q = 0; q < NG; ++q) {
        // (past the end: the last entry's, with zero weights)
        const int e = 16 * q + i;
        const float4 u = *reinterpret_cast<const float4*>(ew + 16LL * (it.y + min(e, n - 1)) + 4 * k);
        w[q][0] = e < n ? u.x : 0.f;
        w[q][1] = e < n ? u.y : 0.f;
        w[q][2] = e < n ? u.z : 0.f;
        w[q][3] = e < n ? u.w : 0.f;
    }
    const int pln = it.x / npp, q0 = it.x - pln * npp;
    const int px0 = (q0 / npy) * pg::kPatch, py0 = (q0 % npy) * pg::kPatch;
    const float2* gp = grids + pln * pstride + (long long)(px0 + k) * Gy + py0;
    const float2* gc[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        const int c = cc * 8 * CT + (CT == 1 ? (i & 7) : 16 * h + i);
        gc[h] = gp + (long long)min(c, nc - 1) * L * G;
    }
    float4 v[2][NH][2];
    float a[2], ai[2];
    auto load = [&](int l, int q) {
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const float4* p = reinterpret_cast<const float4*>(gc[h] + l * G);
            v[q][h][0] = p[0];
            v[q][h][1] = p[1];
        }
        a[q] = AA[(long long)l * M + es];
        if (CPLX) ai[q] = AAi[(long long)l * M + es];
    };
    pg_f4 acc[NG][CT];
#pragma unroll
    for (int q = 0; q < NG; ++q)
#pragma unroll
        for (int t = 0; t < CT; ++t) acc[q][t] = pg_f4{0.f, 0.f, 0.f, 0.f};
    auto sum = [&](int q) {
        // b[t][s]: column i of tile t, point (row k, y = s)
        float b[CT][4];
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const float4 lo = v[q][h][0], hi = v[q][h][1];
            if (CT == 1) {
                const bool im = i >= 8;
                b[0][0] = im ? lo.y : lo.x;
                b[0][1] = im ? lo.w : lo.z;
                b[0][2] = im ? hi.y : hi.x;
                b[0][3] = im ? hi.w : hi.z;
            } else {
                b[(2 * h) % CT][0] = lo.x;
                b[(2 * h) % CT][1] = lo.z;
                b[(2 * h) % CT][2] = hi.x;
                b[(2 * h) % CT][3] = hi.z;
                b[(2 * h + 1) % CT][0] = lo.y;
                b[(2 * h + 1) % CT][1] = lo.w;
                b[(2 * h + 1) % CT][2] = hi.y;
                b[(2 * h + 1) % CT][3] = hi.w;
            }
        }
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (g >= ng) break;
            pg_f4 t4[CT];
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                t4[t] = pg_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    t4[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[g][s], b[t][s], t4[t], 0, 0, 0);
            }
            // times the segment's weight of entry 16 g + 4 k + r
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float ar = __shfl(a[q], 16 * g + 4 * k + r, 64);
#pragma unroll
                for (int t = 0; t < CT; ++t) acc[g][t][r] = __builtin_fmaf(ar, t4[t][r], acc[g][t][r]);
                if constexpr (CPLX) {
                    const float br = __shfl(ai[q], 16 * g + 4 * k + r, 64);
                    if (CT == 1) {
                        // (the other part is 8 columns away: row_ror 8)
                        const float o = __int_as_float(__builtin_amdgcn_update_dpp(
                            0, __float_as_int(t4[0][r]), 0x128, 0xF, 0xF, false));
                        acc[g][0][r] = __builtin_fmaf(i >= 8 ? br : -br, o, acc[g][0][r]);
                    } else {
#pragma unroll
                        for (int h = 0; h < NH; ++h) {
                            const int u = (2 * h) % CT, v1 = (2 * h + 1) % CT;
                            acc[g][u][r] = __builtin_fmaf(-br, t4[v1][r], acc[g][u][r]);
                            acc[g][v1][r] = __builtin_fmaf(br, t4[u][r], acc[g][v1][r]);
                        }
                    }
                }
            }
        }
    };
    // the next segment's values in flight during this one's products (two
    // or three segments ahead measured no faster)
    load(0, 0);
    for (int l = 0; l < L; l += 2) {
        load(min(l + 1, L - 1), 1);
        __builtin_amdgcn_sched_barrier(0);
        sum(0);
        if (l + 1 >= L) break;
        load(min(l + 2, L - 1), 0);
        __builtin_amdgcn_sched_barrier(0);
        sum(1);
    }
    // lane: entries 16 g + 4 k + r, column i of every tile
    float* pp = part + (long long)cc * 16 * CT;
    const long long ps = 16LL * CT * ncc;  // floats per slot
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        if (g >= ng) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = 16 * g + 4 * k + r;
            const long long o = __shfl(sl, e, 64) * ps;
            if (e >= n) continue;
            if constexpr (CT == 1) {
                pp[o + i] = acc[g][0][r];
            } else {
#pragma unroll
                for (int h = 0; h < NH; ++h)
                    *reinterpret_cast<float2*>(pp + o + 32 * h + 2 * i) =
                        make_float2(acc[g][(2 * h) % CT][r], acc[g][(2 * h + 1) % CT][r]);
            }
        }
    }
}

// the samples' sums over their slots soff[i] .. soff[i + 1], in slot order:
// block of 32 samples, lanes over the coils (contiguous), the sums turned
// through LDS into runs of samples.  PLANAR: one chunk of 8 re, then 8 im; else
// a chunk's coils in pairs of floats.
template <bool PLANAR>
__global__ void __launch_bounds__(256) k_interp_sum(const int* __restrict__ soff,
                                                    const float* __restrict__ part, int nc, int rf,
                                                    int M, float2* __restrict__ out,
                                                    long long out_cstride)
{
    // a sample's slots: rows of rf floats; NL lanes of float4 a row
    constexpr int NL = PLANAR ? 4 : 8, NS = 256 / NL;
    __shared__ float buf[4 * NL][NS + 1];
    const int i0 = blockIdx.x * NS, c0 = blockIdx.y * 2 * NL;
    const int s = threadIdx.x / NL, ln = threadIdx.x % NL;
    if (i0 + s < M) {
        const int b = soff[i0 + s], n = soff[i0 + s + 1] - b;
        const float* p = part + (long long)b * rf + 2 * c0 + 4 * ln;
        double t[4] = {0.0, 0.0, 0.0, 0.0};
        // (a window meets at most 9 or 16 patches; six loads in flight)
        for (int q = 0; q < n; q += 6) {
            float4 v[6];
#pragma unroll
            for (int u = 0; u < 6; ++u)
                v[u] = *reinterpret_cast<const float4*>(p + (long long)min(q + u, n - 1) * rf);
#pragma unroll
            for (int u = 0; u < 6; ++u)
                if (q + u < n) {
                    t[0] += v[u].x;
                    t[1] += v[u].y;
                    t[2] += v[u].z;
                    t[3] += v[u].w;
                }
        }
        buf[4 * ln + 0][s] = (float)t[0];
        buf[4 * ln + 1][s] = (float)t[1];
        buf[4 * ln + 2][s] = (float)t[2];
        buf[4 * ln + 3][s] = (float)t[3];
    }
    __syncthreads();
    const int so = threadIdx.x % NS;
#pragma unroll
    for (int co = threadIdx.x / NS; co < 2 * NL; co += NL)
        if (i0 + so < M && c0 + co < nc)
            out[(c0 + co) * out_cstride + i0 + so] =
                PLANAR ? make_float2(buf[co][so], buf[(8 + co) % (4 * NL)][so])
                       : make_float2(buf[2 * co][so], buf[2 * co + 1][so]);
}

// the coil columns of a chunk: one chunk for up to 32 coils (9 or 17 fill about
// half of it), chunks of 32 for more
int interp_mm_width(int nc) { return nc <= 8 ? 8 : nc <= 16 ? 16 : 32; }

void launch_interp_mm(const pg::Gnufft& G, const float2* grids, long long gsz, long long pstride,
                      int nc, int L, int w, const float* AA, const float* AAi, float* part,
                      float2* out, long long out_cstride, hipStream_t s)
{
    const pg::Geometry& g = G.geo;
    const int npy = g.Gy / pg::kPatch, ncc = (nc + w - 1) / w;
    auto launch = [&](auto kern) {
        pg::block_runs(G.n_sblocks, ncc, 64 * kSpreadWaves, [&](int o, int n) {
            hipLaunchKernelGGL(kern, dim3((unsigned)n * ncc * (kSpreadWaves / kIpWaves)),
                               dim3(64 * kIpWaves), 0, s, G.witems + (long long)o * kSpreadWaves,
                               G.entries, G.ent_w, G.islots, npy, grids, gsz, g.Gy, nc, L, AA, AAi,
                               G.M, ncc, part, G.npp, pstride);
        });
    };
    if (AAi)
        w == 8    ? launch(k_interp_mm<1, true>)
        : w == 16 ? launch(k_interp_mm<2, true>)
                  : launch(k_interp_mm<4, true>);
    else
        w == 8    ? launch(k_interp_mm<1, false>)
        : w == 16 ? launch(k_interp_mm<2, false>)
                  : launch(k_interp_mm<4, false>);
    if (w == 8)
        hipLaunchKernelGGL(k_interp_sum<true>, dim3((G.M + 63) / 64), dim3(256), 0, s, G.soff, part,
                           nc, 16, G.M, out, out_cstride);
    else
        hipLaunchKernelGGL(k_interp_sum<false>, dim3((G.M + 31) / 32, (nc + 15) / 16), dim3(256), 0,
                           s, G.soff, part, nc, 2 * ncc * w, G.M, out, out_cstride);
}

// ------------------------------------------- 3-D patch spread ------------
// The full 3-D grid (trajectories that are not stacks of 2-D ones), any
// number of grids.  A wavefront runs the work item items3[] (packed as
// pg_worklist.h says; patch -1: none): it forms a 4x4x4 patch of up
// to 8 NCT grids as a product on the matrix cores,
//   acc[64 points][16 NCT floats] += W[64 points][4 entries] V[4 entries][16 NCT floats]
// four entries a step: per entry the weights wx wy wz of the patch's points,
// formed from the sample's padded weights (wpad), and its row of values
// (re and im as separate columns).  v_mfma_f32_16x16x4f32: A[i][k] in lane
// i + 16k, B[k][j] in lane j + 16k, D[i][j] in lane j + 16 (i / 4), register
// i % 4.  Point tile z holds the patch's plane z, i = 4 x + y; column j of
// float tile t is float NCT j + t of the chunk's row, so a lane loads NCT
// consecutive floats of its entry's row and ends with the 4 points along y
// of plane z and row x = lane / 16.
// Why this form: a thread per grid point (8x8x4 tiles, the values broadcast
// from LDS) left 79% of its lanes outside the sample's window, and the
// central tiles, which every spoke of a radial trajectory crosses, were one
// block's serial loop; here 38% of the products are inside the window, they
// run at the matrix rate (twice the vector one) and patches of more than
// kP3Entries entries are cut into parts, added in part order by
// k_spread3_combine.  32 grids of 128^3, 131072 samples on 1024 spokes: 4860 ->
// 390 us, and 65 us for the parts.  The products themselves take 150 us (128
// clocks per entry and 32 grids) and the 0.8 GB written 170; the rest is the
// latency of each patch's first entries at 3 wavefronts per SIMD.  Runs of four
// patches that no sample meets are stored as whole rows: lane by lane, 32 bytes
// each, the empty part of a large grid took most of a sparse trajectory's time
// (16 grids of 128^3, 1024 samples, whole adjoint: 263 us by the kernel before,
// 390 without the rows, 261 with them).  Few grids
// (a single NUFFT, density compensation) leave columns empty; they took the
// atomic spread before: 6 grids of 60^3, 36080 samples, 11.4 ms -> 0.06 ms
// with the rest of the adjoint.
// Deterministic: entries in sample order, parts in order.  A value that is
// not finite reaches the points of its window alone (a patch's sums are formed
// again then, so it costs others nothing).
constexpr int kP3Waves = 4;

template <int NTP>
__global__ void __launch_bounds__(256) k_wpad3(const float* __restrict__ w, int NT, int M,
                                               float* __restrict__ wpad)
{
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)M * 3 * NTP) return;
    const int i = (int)(e / (3 * NTP)), q = (int)(e - (long long)i * (3 * NTP));
    const int d = q / NTP, j = q - d * NTP - 3;
    wpad[e] = (j >= 0 && j < NT) ? w[(long long)(d * NT + j) * M + i] : 0.f;
}

template <int NTP, int NCT>
__global__ void __launch_bounds__(64 * kP3Waves, NCT == 4 ? 3 : 4) k_spread3(
    const int4* __restrict__ items, const int2* __restrict__ entries,
    const float* __restrict__ wpad, const float2* __restrict__ V, int B,
    float2* __restrict__ grids, long long G, int Gx, int Gy, int npx, int npy,
    float2* __restrict__ partial, int n_slots)
{
    constexpr int CW = 8 * NCT;  // grids per chunk
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int4* bi = items + (long long)blockIdx.x * kP3Waves;
    const int b0 = blockIdx.y * CW;
    bool none = true;
#pragma unroll
    for (int w = 0; w < kP3Waves; ++w) none = none && pg::p3_count(bi[w].z) == 0;
    if (none) {
        // patches (along y) that no sample meets: zeros as whole 128-byte rows,
        // 8 lanes a row, 16 rows (z, x) a grid
        const int4 me = bi[(threadIdx.x & 7) >> 1];
        if (me.x < 0) return;
        const int r = threadIdx.x >> 3 & 15, q = me.x / npx;
        const long long o = ((long long)((q / npy) * 4 + (r >> 2)) * Gx + (me.x % npx) * 4 + (r & 3)) * Gy +
                            (q % npy) * 4 + 2 * (threadIdx.x & 1);
        for (int b = b0 + (int)(threadIdx.x >> 7); b < min(b0 + CW, B); b += kP3Waves / 2)
            *reinterpret_cast<float4*>(grids + b * G + o) = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    const int4 it = bi[wv];
    if (it.x < 0) return;
    const int nf = 2 * min(CW, B - b0);  // floats of the chunk's rows
    const int px = it.x % npx, pr = it.x / npx;
    const int x0 = px * 4, y0 = (pr % npy) * 4, z0 = (pr / npy) * 4;
    const int i = lane & 15, k = lane >> 4;
    const int ax = i >> 2, ay = i & 3;
    // this lane's floats of a row; past the chunk's floats its last ones
    // (those columns are never stored), an odd grid's last pair moved into
    // place (NCT 4, nf % 4 == 2; a last chunk of one grid reads from the grid
    // before it)
    const int fo = min(NCT * i, nf - NCT);
    const bool shifted = NCT == 4 && NCT * i + NCT > nf && NCT * i < nf;
    const float* Vf = reinterpret_cast<const float*>(V) + 2 * (long long)b0 + fo;
    pg_f4 acc[4][NCT];
#pragma unroll
    for (int z = 0; z < 4; ++z)
#pragma unroll
        for (int t = 0; t < NCT; ++t) acc[z][t] = pg_f4{0.f, 0.f, 0.f, 0.f};

    // groups of 4 U entries, the next group's loads in flight during this
    // group's products; the lanes hold 64 entries at a time and the next 64
    // are requested a stage ahead
    constexpr int U = 2, GE = 4 * U, PER = 64 / GE;
    const int n = pg::p3_count(it.z);
    const int ng = (n + GE - 1) / GE;
    float wx[2][U], wy[2][U], v[2][U][NCT];
    pg_f4u wz[2][U];
    int2 cur = make_int2(0, 0), nxt = make_int2(0, 0);
    const int2* ent = entries + pg::p3_first(it.y, it.z);
    auto entry = [&](int st) { return ent[min(64 * st + lane, n - 1)]; };
    auto load_group = [&](int g, int q) {
        if (g % PER == 0) {
            cur = nxt;
            nxt = entry(g / PER + 1);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = (g % PER) * GE + 4 * u + k;
            const int si = __shfl(cur.x, e, 64), sp = __shfl(cur.y, e, 64);
            const float* wp = wpad + (long long)si * (3 * NTP);
            wx[q][u] = wp[(sp & 1023) + ax];
            wy[q][u] = wp[NTP + ((sp >> 10) & 1023) + ay];
            wz[q][u] = *reinterpret_cast<const pg_f4u*>(wp + 2 * NTP + (sp >> 20));
            const float* row = Vf + 2LL * B * si;
            if (NCT == 4) {
                const pg_f4u w = *reinterpret_cast<const pg_f4u*>(row);
#pragma unroll
                for (int t = 0; t < NCT; ++t) v[q][u][t] = w[t];
            } else if (NCT == 2) {
                const pg_f2u w = *reinterpret_cast<const pg_f2u*>(row);
                v[q][u][0] = w[0];
                v[q][u][1 % NCT] = w[1];
            } else {
                v[q][u][0] = row[0];
            }
        }
    };
    auto sum_group = [&](int g, int q) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // entries past the end (the last one again): zero weights and values
            const int m = GE * g + 4 * u + k < n ? -1 : 0;
            const float wxy = __int_as_float(__float_as_int(wx[q][u] * wy[q][u]) & m);
            float vm[NCT];
#pragma unroll
            for (int t = 0; t < NCT; ++t) {
                float w = v[q][u][t];
                if (NCT == 4 && t < 2) w = shifted ? v[q][u][(t + 2) % NCT] : w;
                vm[t] = __int_as_float(__float_as_int(w) & m);
            }
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                const float a = wxy * __int_as_float(__float_as_int(wz[q][u][z]) & m);
#pragma unroll
                for (int t = 0; t < NCT; ++t)
                    acc[z][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vm[t], acc[z][t], 0, 0, 0);
            }
        }
    };
    if (n > 0) {
        nxt = entry(0);
        load_group(0, 0);
        // (groups past the last repeat its entries and add nothing)
        for (int g = 0; g < ng; g += 2) {
            load_group(g + 1, 1);
            __builtin_amdgcn_sched_barrier(0);
            sum_group(g, 0);
            load_group(g + 2, 0);
            __builtin_amdgcn_sched_barrier(0);
            sum_group(g + 1, 1);
        }
    }
    // A value that is not finite has met weights of zero: the points in the
    // windows alone, then, an entry at a time
    bool bad = false;
#pragma unroll
    for (int z = 0; z < 4; ++z)
#pragma unroll
        for (int t = 0; t < NCT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) bad = bad || !(fabsf(acc[z][t][r]) <= FLT_MAX);
    if (__builtin_expect(__any(bad), 0)) {
#pragma unroll
        for (int z = 0; z < 4; ++z)
#pragma unroll
            for (int t = 0; t < NCT; ++t) acc[z][t] = pg_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int e = 0; e < n; ++e) {
            const int2 en = ent[e];
            const float* wp = wpad + (long long)en.x * (3 * NTP);
            const float* row = Vf + 2LL * B * en.x;
            const float wk = wp[(en.y & 1023) + k];
#pragma unroll
            for (int t = 0; t < NCT; ++t) {
                const float w = row[shifted ? (t + 2) % NCT : t];
#pragma unroll
                for (int z = 0; z < 4; ++z)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float q = wk * wp[NTP + ((en.y >> 10) & 1023) + r] *
                                        wp[2 * NTP + (en.y >> 20) + z];
                        if (q != 0.f) acc[z][t][r] += q * w;
                    }
            }
        }
    }
    // lane: points (x0 + k, y0 + r, z0 + z), floats NCT i + t of the chunk
    if (NCT * i >= nf) return;
    if (it.w >= 0) {
        float* pp = reinterpret_cast<float*>(
            partial + ((long long)blockIdx.y * n_slots + it.w) * 64 * CW) + NCT * i;
#pragma unroll
        for (int z = 0; z < 4; ++z)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < NCT; ++t)
                    pp[(z * 16 + k * 4 + r) * 2 * CW + t] = acc[z][t][r];
        return;
    }
    const long long pt = ((long long)z0 * Gx + x0 + k) * Gy + y0;
#pragma unroll
    for (int z = 0; z < 4; ++z) {
        float* gz = reinterpret_cast<float*>(grids + b0 * G + pt + (long long)z * Gx * Gy);
        if (NCT == 1) {
            float* gp = gz + (i >> 1) * 2 * G + (i & 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) gp[2 * r] = acc[z][0][r];
        } else {
            // four points along y: 32 contiguous bytes at a 32-byte boundary
#pragma unroll
            for (int h = 0; h < NCT / 2; ++h) {
                const int gb = (NCT / 2) * i + h;
                if (2 * gb >= nf) break;
                float4* g4 = reinterpret_cast<float4*>(gz + gb * 2 * G);
                const pg_f4 re = acc[z][(2 * h) % NCT], im = acc[z][(2 * h + 1) % NCT];
                g4[0] = make_float4(re[0], im[0], re[1], im[1]);
                g4[1] = make_float4(re[2], im[2], re[3], im[3]);
            }
        }
    }
}

// patches summed in parts: comb = {patch, first slot, parts, 0}; block
// (patch, grid chunk, 256 of its 64 CW sums), the parts added in slot order
template <int CW>
__global__ void __launch_bounds__(256) k_spread3_combine(
    const int4* __restrict__ comb, const float2* __restrict__ partial, int n_slots, int B,
    float2* __restrict__ grids, long long G, int Gx, int Gy, int npx, int npy)
{
    const int4 cb = comb[blockIdx.x];
    const int e = blockIdx.z * 256 + threadIdx.x;
    const int p = e / CW, b = blockIdx.y * CW + e % CW;
    if (b >= B) return;
    const float2* pp = partial + ((long long)blockIdx.y * n_slots + cb.y) * 64 * CW + e;
    float2 t = pp[0];
#pragma unroll 8
    for (int q = 1; q < cb.z; ++q) {
        const float2 v = pp[(long long)q * 64 * CW];
        t.x += v.x;
        t.y += v.y;
    }
    const int px = cb.x % npx, pr = cb.x / npx;
    const int x0 = px * 4, y0 = (pr % npy) * 4, z0 = (pr / npy) * 4;
    grids[b * G + ((long long)(z0 + (p >> 4)) * Gx + x0 + ((p >> 2) & 3)) * Gy + y0 + (p & 3)] = t;
}

template <int NTP>
void launch_spread3(const pg::Gnufft& G, const float2* V, int B, float2* grids, float2* partial,
                    hipStream_t s)
{
    const pg::Geometry& g = G.geo;
    const int npx = g.Gx / 4, npy = g.Gy / 4;
    auto launch = [&](auto kern, auto comb, int cw) {
        const dim3 grid(G.n_items3 / kP3Waves, (B + cw - 1) / cw);
        hipLaunchKernelGGL(kern, grid, dim3(64 * kP3Waves), 0, s, G.items3, G.entries3, G.wpad3, V,
                           B, grids, g.G(), g.Gx, g.Gy, npx, npy, partial,
                           G.n_slots);
        if (G.n_comb > 0)
            hipLaunchKernelGGL(comb, dim3(G.n_comb, grid.y, cw / 4), dim3(256), 0, s, G.comb, partial,
                               G.n_slots, B, grids, g.G(), g.Gx, g.Gy, npx, npy);
    };
    // columns for the grids there are: 8, 16 or (in chunks of) 32
    if (B <= 8)
        launch(k_spread3<NTP, 1>, k_spread3_combine<8>, 8);
    else if (B <= 16)
        launch(k_spread3<NTP, 2>, k_spread3_combine<16>, 16);
    else
        launch(k_spread3<NTP, 4>, k_spread3_combine<32>, 32);
}

// --------------------------------------- atomic spread (one NUFFT at a time)
__global__ void k_zero(float2* __restrict__ p, long long n)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = make_float2(0.f, 0.f);
}

template <int NT, bool D3>
__global__ void __launch_bounds__(256) k_spread_atomic(
    const int* __restrict__ lo, const float* __restrict__ w, int M, int Gx, int Gy, int Gz,
    const float2* __restrict__ in, long long in_cstride, const float2* __restrict__ resid_y,
    const double2* __restrict__ ax64, const float* __restrict__ Wd, int L,
    const float* __restrict__ AA, const float* __restrict__ AAi, int B, float2* __restrict__ grids,
    long long G)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int b = blockIdx.y;
    if (i >= M) return;
    const float2 v = spread_value(in, in_cstride, resid_y, ax64, Wd, AA, AAi, L, M, b, i);
    const int lx = lo[i], ly = lo[M + i], lz = D3 ? lo[2 * M + i] : 0;
    float* g = reinterpret_cast<float*>(grids + (long long)b * G);
    for (int jz = 0; jz < (D3 ? NT : 1); ++jz) {
        const int nz = lz + jz;
        const float wz = D3 ? w[(long long)(2 * NT + jz) * M + i] : 1.f;
        if (D3 && (wz == 0.f || nz < 0 || nz >= Gz)) continue;
        for (int jx = 0; jx < NT; ++jx) {
            const int nx = lx + jx;
            const float wx = w[(long long)jx * M + i];
            if (wx == 0.f || nx < 0 || nx >= Gx) continue;
            for (int jy = 0; jy < NT; ++jy) {
                const int ny = ly + jy;
                const float wy = w[(long long)(NT + jy) * M + i];
                if (wy == 0.f || ny < 0 || ny >= Gy) continue;
                const float ww = D3 ? wx * wy * wz : wx * wy;
                const long long idx = (long long)nz * Gx * Gy + (long long)nx * Gy + ny;
                unsafeAtomicAdd(g + 2 * idx, ww * v.x);
                unsafeAtomicAdd(g + 2 * idx + 1, ww * v.y);
            }
        }
    }
}

template <int NT, bool D3>
void interp_dispatch(const pg::Gnufft& G, const float2* grids, int nc, int L, const float* AA,
                     const float* AAi, float2* out, long long out_cstride, hipStream_t s,
                     bool planes, float* part, size_t part_cap)
{
    const pg::Geometry& g = G.geo;
    const pg::Gnufft::Tuned* tn = G.tuned_for(nc, L, AAi != nullptr);
    // z-class planes: a 2-D interpolation on the plane of each sample's class
    const long long gsz = planes ? (long long)g.Gx * g.Gy : g.G();
    const long long pstride = planes ? (long long)nc * L * gsz : 0;
    const int v4 = pgk::g_interp4.load(std::memory_order_relaxed);
    if ((!D3 || planes) && part && pgk::interp_mm_possible(G, nc, L, AA != nullptr, part_cap) &&
        (tn ? tn->mm : v4 == 3 || (v4 == 1 && pgk::interp_mm_pays(G, nc, L, AAi != nullptr)))) {
        launch_interp_mm(G, grids, gsz, pstride, nc, L, interp_mm_width(nc), AA, AAi, part, out,
                         out_cstride, s);
        return;
    }
    if ((!D3 || planes) && NT <= 8 && pgk::interp_lds_possible(G, L, AA != nullptr) &&
        (!tn || tn->lds)) {
        // four segments per stage when the autotuner chose it, or else from
        // four segments up (measured faster there: the smaller blocks and
        // LDS footprint keep more of them per CU)
        const bool four = tn ? tn->lds == 2 : (v4 == 2 || (v4 != 0 && L >= 4));
        // (its staging and weight offsets are 32-bit byte offsets)
        if (G.n_iitems4 > 0 && four && gsz * 4 * 8 < (1LL << 31) &&
            (long long)L * G.M * 4 < (1LL << 31)) {
            auto launch = [&](auto kern) {
                pg::coil_runs(nc, G.n_iitems4, kI4Threads, [&](int c, int n) {
                    hipLaunchKernelGGL(kern, dim3((unsigned)G.n_iitems4 * n), dim3(kI4Threads), 0, s,
                                       G.iitems4, G.irec4, G.ity, G.ipadl, grids + c * L * gsz, gsz,
                                       g.Gx, g.Gy, n, L, AA, AAi, G.M, out + c * out_cstride,
                                       out_cstride, pstride);
                });
            };
            AAi ? launch(k_interp_lds4<true>) : launch(k_interp_lds4<false>);
            return;
        }
        auto launch = [&](auto kern) {
            pg::coil_runs(nc, G.n_iitems, 64 * kInterpWaves, [&](int c, int n) {
                hipLaunchKernelGGL(kern, dim3((unsigned)G.n_iitems * n), dim3(64 * kInterpWaves), 0,
                                   s, G.iitems, G.irec, G.ity, G.ipadl, grids + c * L * gsz, gsz,
                                   g.Gx, g.Gy, n, L, AA, AAi, G.M, out + c * out_cstride,
                                   out_cstride, pstride);
            });
        };
        if (L <= 8)
            AAi ? launch(k_interp_lds<8, true>) : launch(k_interp_lds<8, false>);
        else
            AAi ? launch(k_interp_lds<16, true>) : launch(k_interp_lds<16, false>);
        return;
    }
    const int nsb = (G.M + 63) / 64;  // 64 samples (4 lanes each) per block
    auto gather = [&](auto kern, int Gz, const int* zcls) {
        pg::coil_runs(nc, nsb, 256, [&](int c, int n) {
            hipLaunchKernelGGL(kern, dim3((unsigned)nsb * n), dim3(256), 0, s, G.lo, G.w, G.M, g.Gx,
                               g.Gy, Gz, grids + c * L * gsz, gsz, n, L, AA, AAi,
                               out + c * out_cstride, out_cstride, nsb, n % 8 == 0 ? 1 : 0, zcls,
                               pstride);
        });
    };
    if (planes) return gather(k_interp<NT, false>, 1, G.zcls);
    if constexpr (D3 && NT <= 8) {
        // A tile costs a block and its whole region whatever it holds, and one
        // or two segments hide little of its loads: where such a batch has more
        // blocks than run at a time and few samples in each, the gather is the
        // faster form (a multiple of 8 coils, each on its XCD's L2, somewhat
        // earlier).  Spokes of 64 samples, tiles / gather in us: 128^3, 256
        // spokes (2.6 samples a tile) 1 grid 114 / 95, 4 grids 465 / 392, 2 coils x 2
        // segments 441 / 394, 1 x 4 432 / 451; 64 spokes 2 x 2 359 / 377; 64^3, 64
        // spokes (4.6) 1 grid 30 / 41, 8 grids 106 / 90, 17 grids 260 / 270; 256 spokes
        // (7.9) 1 grid 38 / 43, 4 grids 88 / 107, 8 grids 162 / 154.
        const bool sparse = L <= 2 && (long long)G.n_iitems3 * nc * L >= (L == 1 ? 4096 : 16384) &&
                            G.M < (nc % 8 ? 6LL : 8LL) * G.n_iitems3;
        // (32-bit byte offsets within a grid)
        if (G.n_iitems3 > 0 && !sparse && g.G() * 8 < (1LL << 31)) {
            const int per = (G.n_iitems3 + 7) / 8;
            auto launch = [&](auto kern) {
                pg::coil_runs(nc, 8 * per, 8 * kI3Chunk, [&](int c, int n) {
                    hipLaunchKernelGGL(kern, dim3((unsigned)(8 * per * n)), dim3(8 * kI3Chunk), 0, s,
                                       G.iitems3, G.n_iitems3, G.irec3, G.wpad3, G.itx, G.ity,
                                       G.ipadl, grids + c * L * gsz, gsz, g.Gx, g.Gy, g.Gz, n, L, AA,
                                       AAi, G.M, out + c * out_cstride, out_cstride, per);
                });
            };
            AAi ? launch(k_interp3_lds<NT, true>) : launch(k_interp3_lds<NT, false>);
            return;
        }
    }
    gather(k_interp<NT, D3>, g.Gz, nullptr);
}

template <int NT, bool D3>
void spread_dispatch(const pg::Gnufft& G, const float2* in, long long in_cstride, int nc, int L,
                     const float* AA, const float* AAi, const float2* resid_y, const double2* ax64,
                     const float* Wd, float2* grids, bool vals_ready, hipStream_t s, bool planes,
                     float2* vals, float2* partial)
{
    const pg::Geometry& g = G.geo;
    const int B = nc * L;
    if (D3 && !planes && G.nzc > 0) {
        // a plan of z-class planes has no 3-D work lists
        const long long n = (long long)B * g.G();
        hipLaunchKernelGGL(k_zero, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, grids, n);
        hipLaunchKernelGGL((k_spread_atomic<NT, D3>), dim3((G.M + 255) / 256, B), dim3(256), 0, s,
                           G.lo, G.w, G.M, g.Gx, g.Gy, g.Gz, in, in_cstride, resid_y, ax64, Wd, L,
                           AA, AAi, B, grids, g.G());
        return;
    }
    // per-sample values of every grid (or the compact rows they are formed
    // from), once
    const int S = pgk::spread_row_floats(G, nc, L, AA, AAi);
    if (!vals_ready) {
        if (S)
            launch_rows(in, in_cstride, resid_y, ax64, Wd, L, AA, AAi, G.M, nc, S, vals, s);
        else
            launch_values(in, in_cstride, resid_y, ax64, Wd, L, AA, AAi, G.M, B, vals, s);
    }
    if (!D3 || planes) {
        // 2-D patches (of every z-class plane); plane p of grid b at
        // (p*B + b)*Gx*Gy
        const long long gsz = planes ? (long long)g.Gx * g.Gy : g.G();
        const long long pstride = planes ? (long long)B * gsz : 0;
        const float* rows = reinterpret_cast<const float*>(vals);
        if (S)
            launch_spread2(G, rows, S, nc, L, AAi ? 2 : 1, grids, gsz, pstride, partial, s);
        else
            launch_spread2(G, rows, 2 * B, B, 1, 0, grids, gsz, pstride, partial, s);
        return;
    }
    if (NT == 12)
        launch_spread3<20>(G, vals, B, grids, partial, s);
    else
        launch_spread3<16>(G, vals, B, grids, partial, s);
}

}  // namespace

namespace pgk {

std::atomic<int> g_zclass{1};
std::atomic<int> g_interp4{1};
std::atomic<int> g_spread_rows{1};
std::atomic<int> g_zfuse{1};
std::atomic<int> g_zmfma{1};
std::atomic<int> g_zamfma{1};
std::atomic<int> g_zfwd{1};

int spread_row_floats(const pg::Gnufft& G, int nc, int L, const float* AA, const float* AAi)
{
    const int B = nc * L;
    if (!g_spread_rows.load(std::memory_order_relaxed) || !AA || L < 2) return 0;
    if (G.geo.dims == 3 && !zclass_active(G, B)) return 0;
    // Value rows where the compact ones leave columns of the products empty: a
    // tile of 16 columns holds 8 coils of one segment there, here 8 grids of any.
    // They are more memory to write and read, so a fifth of the tiles has to be
    // saved, past 64 grids a third and the values have to stay in the caches.
    // Adjoint, compact / value rows (us): 1 coil x 8 segments, 512^2, 8192
    // samples 125 / 91 (101 with a lane per grid), 3 x 5 229 / 183 (197); 128^2,
    // 32768 samples: 1 x 8 42 / 27, 11 x 5 70 / 62, 9 x 4 (as many tiles) 53.5 / 55.2;
    // 17 x 12 (53 MB of values) 161 / 146, 192^2, 65536 samples (107 MB) 340 / 356.
    auto tiles = [](int cols) { return cols <= 8 ? 1 : cols <= 16 ? 2 : 4 * ((cols + 31) / 32); };
    const int tv = tiles(B), tc = tiles(nc) * L;
    if (B <= 64 ? 5 * tv <= 4 * tc : 3 * tv <= 2 * tc && 8.0 * G.M * B <= 54e6) return 0;
    const int S = (2 * nc + (AAi ? 2 : 1) * L + 3) & ~3;
    // the rows live in the plan's value buffer (M x B float2) and a block of
    // 64 rows in LDS
    return (S <= 2 * B && S <= 128) ? S : 0;
}

bool zclass_active(const pg::Gnufft& G, int B)
{
    return G.nzc > 0 && B >= 16 && (long long)B * G.nzc < (1LL << 31);
}

// The batches that the patch interpolation can take: 8 coils (fewer leave
// matrix columns idle), 6 segments (a partial sum is written and read once for
// all of them) and 64 grids, patches of 16 entries on the average (one group
// of the products), and partial sums that fit part_cap floats.
bool interp_mm_possible(const pg::Gnufft& G, int nc, int L, bool aa, size_t part_cap)
{
    if (!aa || !G.islots || nc < 8 || L < 6 || nc * L < 64) return false;
    const size_t patches = (size_t)G.npp * (G.nzc > 0 ? G.nzc : 1);
    const int w = interp_mm_width(nc);
    return G.n_entries >= pg::kIpEntries * patches && G.n_entries * 2 * ((nc + w - 1) / w * w) <= part_cap;
}

// Which of them it is the faster form for.  Against it are a wavefront's
// serial chain over the segments (some 1 us each while the patches' wavefronts
// do not fill the SIMDs), columns without a coil, the launch of the second pass
// and, for up to 8 coils, whose products are short, the shuffles of the weights
// (complex ones above all); the tiled form pays for segments in fours (L4).  So
// patches x sqrt(entries a patch) x (filled share of the columns)^2 x L4^2 / L
// has to exceed a bound.  5687 random batches (48^2 .. 256^2 and stacks of 32^2
// .. 64^2, 8 .. 32 coils, 6 .. 12 segments, whole forward operator): patches in
// 0.63 to 1.43 times the tiles' time, over 1.05 in 1371.  Of the 3720 that pass
// the bound 34 are slower by over 5%; 59 of the others would gain as much.  128^2, 32768 samples, 8 coils x 8 segments: 56.8 (tiles) / 56.6
// us, 32 x 12: 265 / 210; 64^2, 4096 samples, 17 x 8: 34.0 / 47.8.  Batches that
// have no tiles (12 taps, over 16 segments) would go to the gather kernel.
bool interp_mm_pays(const pg::Gnufft& G, int nc, int L, bool cplx)
{
    if (!interp_lds_possible(G, L, true)) return true;
    const int w = interp_mm_width(nc), l4 = (L + 3) & ~3;
    const double patches = (double)G.npp * (G.nzc > 0 ? G.nzc : 1);
    const double fill = (double)nc / ((nc + w - 1) / w * w);
    double bound = 8e4;
    if (w == 8) bound *= 1.5;
    if (cplx) bound *= w == 8 ? 2.0 : 1.125;
    return std::sqrt(patches * G.n_entries) * fill * fill * l4 * l4 >= bound * L;
}

bool interp_lds_possible(const pg::Gnufft& G, int L, bool aa)
{
    const pg::Geometry& g = G.geo;
    return (g.dims == 2 || G.nzc > 0) && g.ntaps <= 8 && aa && L >= 2 && L <= 16 &&
           G.n_iitems > 0 && (long long)L * g.Gx * g.Gy < (1LL << 31);
}

void launch_interp(const pg::Gnufft& G, const float2* grids, int nc, int L, const float* AA,
                   const float* AAi, float2* out, long long out_cstride, hipStream_t s, bool planes,
                   float* part, size_t part_cap)
{
    PG_REQUIRE(!planes || zclass_active(G, nc * L), PG_ERR_STATE, "no z-class planes for this batch");
    const bool d3 = G.geo.dims == 3;
    switch (G.geo.ntaps) {
    case 8:
        d3 ? interp_dispatch<8, true>(G, grids, nc, L, AA, AAi, out, out_cstride, s, planes, part, part_cap)
           : interp_dispatch<8, false>(G, grids, nc, L, AA, AAi, out, out_cstride, s, planes, part, part_cap);
        break;
    case 6:
        d3 ? interp_dispatch<6, true>(G, grids, nc, L, AA, AAi, out, out_cstride, s, planes, part, part_cap)
           : interp_dispatch<6, false>(G, grids, nc, L, AA, AAi, out, out_cstride, s, planes, part, part_cap);
        break;
    case 12:
        d3 ? interp_dispatch<12, true>(G, grids, nc, L, AA, AAi, out, out_cstride, s, planes, part, part_cap)
           : interp_dispatch<12, false>(G, grids, nc, L, AA, AAi, out, out_cstride, s, planes, part, part_cap);
        break;
    default:
        throw pg::Error{PG_ERR_UNSUPPORTED, "kernel width * gridos must give 6, 8 or 12 taps"};
    }
}

bool spread_uses_values(const pg::Gnufft& G, int B)
{
    return G.geo.dims == 2 || G.nzc == 0 || zclass_active(G, B);
}

void build_wpad3(const pg::Gnufft& G, hipStream_t s)
{
    const int ntp = pg::wpad3_len(G.geo.ntaps);
    const long long n = (long long)G.M * 3 * ntp;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (ntp == 20)
        hipLaunchKernelGGL(k_wpad3<20>, grid, dim3(256), 0, s, G.w, G.geo.ntaps, G.M, G.wpad3);
    else
        hipLaunchKernelGGL(k_wpad3<16>, grid, dim3(256), 0, s, G.w, G.geo.ntaps, G.M, G.wpad3);
}

void launch_spread_values(const pg::Gnufft& G, const float2* in, long long in_cstride, int nc,
                          int L, const float* AA, const float* AAi, const float2* resid_y,
                          const double2* ax64, const float* Wd, hipStream_t s, float2* vals)
{
    const int S = spread_row_floats(G, nc, L, AA, AAi);
    if (S)
        launch_rows(in, in_cstride, resid_y, ax64, Wd, L, AA, AAi, G.M, nc, S, vals ? vals : G.vals,
                    s);
    else
        launch_values(in, in_cstride, resid_y, ax64, Wd, L, AA, AAi, G.M, nc * L,
                      vals ? vals : G.vals, s);
}

void launch_spread(const pg::Gnufft& G, const float2* in, long long in_cstride, int nc, int L,
                   const float* AA, const float* AAi, const float2* resid_y, const double2* ax64,
                   const float* Wd, float2* grids, bool vals_ready, hipStream_t s, bool planes,
                   float2* vals, float2* partial)
{
    PG_REQUIRE(!planes || zclass_active(G, nc * L), PG_ERR_STATE, "no z-class planes for this batch");
    if (!vals) vals = G.vals;
    if (!partial) partial = G.partial;
    const bool d3 = G.geo.dims == 3;
    switch (G.geo.ntaps) {
    case 8:
        d3 ? spread_dispatch<8, true>(G, in, in_cstride, nc, L, AA, AAi, resid_y, ax64, Wd,
                                      grids, vals_ready, s, planes, vals, partial)
           : spread_dispatch<8, false>(G, in, in_cstride, nc, L, AA, AAi, resid_y, ax64, Wd,
                                       grids, vals_ready, s, planes, vals, partial);
        break;
    case 6:
        d3 ? spread_dispatch<6, true>(G, in, in_cstride, nc, L, AA, AAi, resid_y, ax64, Wd,
                                      grids, vals_ready, s, planes, vals, partial)
           : spread_dispatch<6, false>(G, in, in_cstride, nc, L, AA, AAi, resid_y, ax64, Wd,
                                       grids, vals_ready, s, planes, vals, partial);
        break;
    case 12:
        d3 ? spread_dispatch<12, true>(G, in, in_cstride, nc, L, AA, AAi, resid_y, ax64, Wd,
                                       grids, vals_ready, s, planes, vals, partial)
           : spread_dispatch<12, false>(G, in, in_cstride, nc, L, AA, AAi, resid_y, ax64, Wd,
                                        grids, vals_ready, s, planes, vals, partial);
        break;
    default:
        throw pg::Error{PG_ERR_UNSUPPORTED, "kernel width * gridos must give 6, 8 or 12 taps"};
    }
}

}  // namespace pgk
