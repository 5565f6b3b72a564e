// GPU kernels of the Monte Carlo radiative-transfer solver (gfx950).
//
//   raygen_plain   Philox rays: (band, g) from the Tmax proposal, isotropic
//                  direction uniforms, bundle weights -> SoA descriptors.
//   raygen_compat  reference sampling: XORWOW stream per (cell, block) for
//                  (band, g), Sobol32 dims 0/1 for directions.
//   trace          persistent cell-by-cell traversal (code/mc_gpu.cu:228-438)
//                  with FP64 per-slot tallies.
//   reduce_rays    deterministic per-slot sum of per-ray tallies (FP64, Kahan
//                  FP32 or plain FP32).
//   spline_pass    one axis of the natural-spline coarse-grid interpolation
//                  (code/spline.cpp:35-116).
//   finalize       Q = E - A, standard error (code/mc_gpu.cu:212-222).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dmath.h"
#include "kernels.h"
#include "../../include/dnsmc_rad.h"

namespace dn {

typedef __attribute__((address_space(1))) const float gfloat;

// Emitter weights shared by the generators: Ibmax kappa_i Ib_i / (kappa_max Ib_max)
// (code/mc_gpu.cu:63,:163-169).
__device__ __forceinline__ void bundle_weight(const GenArgs& a, const float* ib_tab, float Ti, int band, int g,
                                              float* w, float* winv, float* inv_ib)
{
    float kap, ib;
    int bg = band * a.nQ + g;
    if (a.spec == kSpecGreyT4) {
        float t2 = Ti * Ti;
        kap = a.kappa_grey;
        ib = t2 * t2;
    } else {
        float pos = fmaf(Ti, a.inv_dT, a.mT0);
        pos = fminf(fmaxf(pos, 0.0f), (float)(a.nT - 1));
        int t0 = (int)pos;
        t0 = t0 > a.nT - 2 ? a.nT - 2 : t0;
        float fr = pos - (float)t0;
        const float* kr = a.kq + (size_t)bg * a.nT;
        float k0 = kr[t0], k1 = kr[t0 + 1];
        kap = fmaf(fr, k1 - k0, k0);
        const float* ir = ib_tab + (size_t)band * a.nT;
        float i0 = ir[t0], i1 = ir[t0 + 1];
        ib = fmaf(fr, i1 - i0, i0);
    }
    float ww = a.Ibmax * (kap * ib) * a.inv_emax[bg];
    *w = ww;
    *inv_ib = 1.0f / ib;
    *winv = ww * *inv_ib;
}

// ------------------------------------------------------- raygen_plain ----
// One thread per ray.  Counter (r, cell, snapshot, 0), key = seed: the draw of
// a ray depends only on its identity, not on the launch shape.
__global__ __launch_bounds__(256) void raygen_plain(GenArgs a)
{
    extern __shared__ float lds[];
    float* s_cdfb = lds;
    float* s_cdfg = s_cdfb + a.nB;
    float* s_ib = s_cdfg + a.nB * a.nQ;
    const bool ib_lds = a.spec == kSpecTable && a.nB * a.nT <= 16384;
    for (int i = threadIdx.x; i < a.nB; i += blockDim.x) s_cdfb[i] = a.cdf_band[i];
    for (int i = threadIdx.x; i < a.nB * a.nQ; i += blockDim.x) s_cdfg[i] = a.cdf_g[i];
    if (ib_lds)
        for (int i = threadIdx.x; i < a.nB * a.nT; i += blockDim.x) s_ib[i] = a.Ib[i];
    __syncthreads();
    const float* ibt = ib_lds ? s_ib : a.Ib;
    const long long nr = a.nslots * (long long)a.rays_per_slot;
    for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < nr; q += (long long)gridDim.x * blockDim.x) {
        long long sl = q / a.rays_per_slot;
        int r = (int)(q - sl * a.rays_per_slot);
        const int4 si = a.slotinfo[a.slot0 + sl];
        const int cell = si.y;
        u32x4 x = philox4x32_10(u32x4{(uint32_t)r, (uint32_t)cell, (uint32_t)a.snap, 0u}, (uint32_t)a.seed,
                                (uint32_t)(a.seed >> 32));
        int band = cdf_search(s_cdfb, a.nB, u01_open(x.x));
        int g = a.g_search ? cdf_search(s_cdfg + band * a.nQ, a.nQ, u01_open(x.y)) : 0;
        g = g > a.nQ - 1 ? a.nQ - 1 : g;
        float Ti = a.T0[(size_t)a.snap * a.tstride0 + si.z];
        float w, winv, iib;
        bundle_weight(a, ibt, Ti, band, g, &w, &winv, &iib);
        uint32_t w0, w1;
        desc_pack(x.z >> 8, x.w >> 8, band, g, &w0, &w1);
        a.w0[q] = w0;
        a.w1[q] = w1;
        a.w[q] = w;
        a.winv[q] = winv;
    }
}

// ------------------------------------------------------ raygen_compat ----
__device__ __forceinline__ uint32_t sobol_at(const uint32_t* v, uint64_t n)
{
    const uint32_t gc = (uint32_t)(n ^ (n >> 1));
    uint32_t x = 0;
#pragma unroll 8
    for (int k = 0; k < 32; ++k) x ^= v[k] & (uint32_t)((int32_t)(gc << (31 - k)) >> 31);
    return x;
}

// Exclusive or over the wave, in every lane.
__device__ __forceinline__ uint32_t wave_xor(uint32_t v)
{
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);    // quad: lane ^ 1
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false);    // quad: lane ^ 2
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false);   // row_half_mirror
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, false);   // row_mirror
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0) ^ (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    return a ^ (uint32_t)__builtin_amdgcn_readlane((int)v, 32) ^ (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
}

// XORWOW stream of a compat slot (cell, block v), seeded as
// curand_init(1234, subsequence, 0) is in code/mc_gpu.cu:99: own seed
// scramble, subsequence = the reference's product
// (idx+1)(stream+1)(v+1)(1+gpu)ystart over its stream decomposition of the
// cell (code/mc_gpu.cu:84-87), jump 2^67 per subsequence.
//
// The generator's recurrence is linear over GF(2) with step matrix A, and its
// state after i steps is y_i .. y_{i+4} of one word sequence.  Called by one
// wave: the subsequence's 160 x 160 bit matrices are applied to the seed with
// 64 columns at a time across the lanes, and the first kXwSeq words of the
// slot's sequence are written to y.  Threads then start anywhere in the stream
// with one product, xorwow_jump.
__device__ __forceinline__ void compat_sequence(const GenArgs& a, int cell, int v, int lane, uint32_t* y)
{
    int ci = cell % a.n0, cj = (cell / a.n0) % a.n1, ck = cell / (a.n0 * a.n1);
    int per_stream = a.n0 / a.num_streams;
    int stream = ci / per_stream;
    int jloc = cj - (a.ystart - 1);
    int kloc = ck - a.gpu * (a.n2 / a.num_gpu);
    int idx = (ci - stream * per_stream) * (a.n2 / a.num_gpu * (a.n1 / a.p_row)) + jloc * (a.n2 / a.num_gpu) + kloc;
    int32_t prod = (int32_t)((uint32_t)(idx + 1) * (uint32_t)(stream + 1) * (uint32_t)(v + 1) *
                             (uint32_t)(1 + a.gpu) * (uint32_t)a.ystart);
    prod = __builtin_amdgcn_readfirstlane(prod);
    uint64_t m = (uint64_t)(int64_t)prod & ((1ull << 60) - 1ull);
    uint32_t x[5];
    for (int w = 0; w < 5; ++w) x[w] = a.xw_seed[w];
    const uint32_t* col = a.xw_jump_sub + lane * 5;
    const int l5 = lane & 31;
    uint32_t c[15], d[15];
    auto load = [&](int j, uint32_t* o) {   // columns lane, lane + 64 and (lanes 0..31) lane + 128
        const uint32_t* q = col + (size_t)j * 800;
#pragma unroll
        for (int w = 0; w < 5; ++w) {
            o[w] = q[w];
            o[5 + w] = q[320 + w];
            o[10 + w] = q[lane < 32 ? 640 + w : w];
        }
    };
    if (m) load(__builtin_ctzll(m), c);
    while (m) {
        m &= m - 1;
        if (m) load(__builtin_ctzll(m), d);
        const uint32_t m0 = 0u - (((lane < 32 ? x[0] : x[1]) >> l5) & 1u);
        const uint32_t m1 = 0u - (((lane < 32 ? x[2] : x[3]) >> l5) & 1u);
        const uint32_t m2 = lane < 32 ? 0u - ((x[4] >> l5) & 1u) : 0u;
#pragma unroll
        for (int w = 0; w < 5; ++w) x[w] = wave_xor((c[w] & m0) ^ (c[5 + w] & m1) ^ (c[10 + w] & m2));
#pragma unroll
        for (int w = 0; w < 15; ++w) c[w] = d[w];
    }
    Xorwow s{x[0], x[1], x[2], x[3], x[4], 0u};
    if (lane < 5) y[lane] = lane == 0 ? x[0] : lane == 1 ? x[1] : lane == 2 ? x[2] : lane == 3 ? x[3] : x[4];
#pragma unroll 5
    for (int i = 5; i < kXwSeq; ++i) {
        (void)xorwow_next(s);
        if (lane == 0) y[i] = s.x4;
    }
}

// State n steps into the stream: A^n = sum of c_i A^i, i < 160, with
// c = x^n modulo A's characteristic polynomial (the host's table), so the
// state is the sum of the c_i = 1 states of the sequence y.
__device__ __forceinline__ Xorwow xorwow_jump(const uint32_t* y, const uint32_t* poly, uint32_t d0, uint32_t n)
{
    uint32_t r[5] = {0, 0, 0, 0, 0}, c[5];
#pragma unroll
    for (int w = 0; w < 5; ++w) c[w] = poly[w];
    uint4 lo = *(const uint4*)y;
#pragma unroll 1
    for (int j = 0; j < 5; ++j) {
#pragma unroll
        for (int i = 0; i < 32; i += 4) {
            const uint4 hi = *(const uint4*)(y + 32 * j + i + 4);
            const uint32_t q[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t m = (uint32_t)((int32_t)(c[0] << (31 - (i + b))) >> 31);
#pragma unroll
                for (int w = 0; w < 5; ++w) r[w] = __builtin_amdgcn_bitop3_b32(m, q[b + w], r[w], 0x6A);   // r ^ (m & q)
            }
            lo = hi;
        }
        c[0] = c[1]; c[1] = c[2]; c[2] = c[3]; c[3] = c[4];
    }
    return Xorwow{r[0], r[1], r[2], r[3], r[4], d0 + 362437u * n};
}

// One block per slot, the bundles in runs of run_len consecutive ones per
// thread (at most one run each).  The Sobol points are v*photmax + h (the Sobol
// states restart per cell, :79-82).  Descriptors are staged in LDS, kStage
// bundles of every run at a time, and leave in pieces of 64 (32) bytes; the
// weights of the slot's (band, g) bins are computed once where a slot has at
// least as many bundles as bins.
//
// Before, each thread of 256 bundles multiplied the seed by its subsequence's
// and offset's matrices alone, 160 columns of five words at a time.  A solve of
// 9216 slots of 1019 bundles went from 1.76 to 1.06 ms with this kernel.
__global__ __launch_bounds__(256) void raygen_compat(GenArgs a)
{
    extern __shared__ __align__(16) float lds[];
    const int nbin = a.nB * a.nQ, tid = threadIdx.x, nth = blockDim.x;
    const int R = a.rays_per_slot, L = a.run_len;
    const int st = L < 16 ? 8 : 16, sh = L < 16 ? 3 : 4;   // staged bundles per run (divides L)
    uint32_t* s_y = (uint32_t*)lds;
    uint32_t* s_sob = s_y + kXwSeq;
    uint32_t* s_w0 = s_sob + 64;
    uint32_t* s_w1 = s_w0 + nth * (st + 1);
    float* s_cdfb = (float*)(s_w1 + nth * (st + 1));
    float* s_iib = s_cdfb + a.nB;
    float* s_bw = s_iib + a.nB;                            // weight of each bin (bin_weights)
    float* s_cdfg = s_bw + (a.bin_weights ? nbin : 0);
    const float* cdfg = a.cdf_lds ? s_cdfg : a.cdf_g;
    for (int i = tid; i < a.nB; i += nth) s_cdfb[i] = a.cdf_band[i];
    if (a.cdf_lds)
        for (int i = tid; i < nbin; i += nth) s_cdfg[i] = a.cdf_g[i];
    for (int i = tid; i < 64; i += nth) s_sob[i] = a.sobol_v[i];
    const int h0 = tid * L;
    for (long long sl = blockIdx.x; sl < a.nslots; sl += gridDim.x) {
        const int4 si = a.slotinfo[a.slot0 + sl];
        const int cell = si.y;
        const int v = si.x % a.slots_per_emitter;
        const float Ti = a.T0[(size_t)a.snap * a.tstride0 + si.z];
        if (tid < 64) compat_sequence(a, cell, v, tid, s_y);
        if (a.bin_weights)
            for (int k = tid; k < nbin; k += nth) {
                const int band = (int)fdiv((uint32_t)k, a.fd_nQ), g = k - band * a.nQ;
                float w, winv, iib;
                bundle_weight(a, a.Ib, Ti, band, g, &w, &winv, &iib);
                s_bw[k] = w;
                if (g == 0) s_iib[band] = iib;
            }
        __syncthreads();
        Xorwow s{0, 0, 0, 0, 0, 0};
        uint32_t sx0 = 0, sx1 = 0;
        uint64_t n = (uint64_t)v * (uint64_t)R + (uint64_t)h0;
        if (h0 < R) {
            s = xorwow_jump(s_y, a.xw_poly + 5 * tid, a.xw_seed[5], (uint32_t)h0 * (uint32_t)a.draws_per_bundle);
            if (a.use_sobol) {
                sx0 = sobol_at(s_sob, n);
                sx1 = sobol_at(s_sob + 32, n);
            }
        }
        for (int b0 = 0; b0 < L; b0 += st) {
            if (b0 > 0) __syncthreads();
            for (int i = 0; i < st && h0 + b0 + i < R; ++i) {
                uint32_t mp, mt;
                if (a.use_sobol) {
                    mp = sx0 >> 8;
                    mt = sx1 >> 8;
                    int c = __builtin_ctzll(~n);
                    sx0 ^= s_sob[c];
                    sx1 ^= s_sob[32 + c];
                    ++n;
                } else {
                    mp = xorwow_next(s) >> 8;
                    mt = xorwow_next(s) >> 8;
                }
                int band = cdf_search(s_cdfb, a.nB, u01_incl(xorwow_next(s)));
                int g = 0;
                if (a.g_search) g = cdf_search(cdfg + band * a.nQ, a.nQ, u01_incl(xorwow_next(s)));
                g = g > a.nQ - 1 ? a.nQ - 1 : g;
                desc_pack(mt, mp, band, g, &s_w0[tid * (st + 1) + i], &s_w1[tid * (st + 1) + i]);
            }
            __syncthreads();
            for (int e = tid; e < nth << sh; e += nth) {
                const int t = e >> sh, i = e & (st - 1), h = t * L + b0 + i;
                if (h < R) {
                    const uint32_t w0 = s_w0[t * (st + 1) + i], w1 = s_w1[t * (st + 1) + i];
                    const int band = desc_band(w0, w1), g = desc_g(w1);
                    float w, winv, iib;
                    if (a.bin_weights) {
                        w = s_bw[band * a.nQ + g];
                        winv = w * s_iib[band];
                    } else {
                        bundle_weight(a, a.Ib, Ti, band, g, &w, &winv, &iib);
                    }
                    const long long q = sl * R + h;
                    a.w0[q] = w0;
                    a.w1[q] = w1;
                    a.w[q] = w;
                    a.winv[q] = winv;
                }
            }
        }
        __syncthreads();   // the next slot's sequence and weights
    }
}

// Sorted compat generation (srt == 1: code/mc_gpu.cu:100-102, :138-139).  The
// reference draws all photmax (band, g) pairs of the slot's stream first and
// counts them (kernel_find, :786-812), then replays the counts position by
// position of the kavg band order, g ascending inside a band (wave_find,
// :897-930), drawing each bundle's direction in the photon loop.  Bundles with
// the same (band, g) are interchangeable until a direction is attached, so
// the replay is a histogram and a scan: one block per slot,
//  (1) each thread jumps to its run of (band, g) draws and counts them in LDS,
//  (2) the histogram is scanned in replay order (position p, then g), and each
//      drawn bin's weights take the place of its count and CDF entry,
//  (3) bundle h takes the bin where the running count first exceeds h, and its
//      direction is Sobol point v*photmax + h, or XORWOW uniforms
//      draws_find*photmax + 2h (phi) and + 2h + 1 (theta) of the stream.
// The reference permutes its tables into the sorted order, so position p
// carries band band_order[p]; the descriptor holds that band.
//
// (3) gives each wave 64 consecutive bundles at a time, so the four arrays are
// written in whole lines, and finds the bins by walking the running counts, a
// lane each, once for the 64.  With Sobol directions the 64 start at a multiple
// of 64 of the sequence: a point is then the exclusive or of the wave's (one
// step per 64) and the lane's (constant) part.
//
// 3.7e8 bundles of 18432 slots (100 bands x 16 g): 20.9 -> 3.2 ms (the 16 B per
// bundle alone 1 ms; instruction issue and the two CDF searches' LDS reads bound
// it).  Before, every thread multiplied its slot's seed by the subsequence's and
// its offset's bit matrices alone, weights were computed and tables gathered per
// bundle, and the lanes of a wave wrote 64 different lines.  Seven blocks per CU
// (LDS) against five and six with more registers: 3.2, 4.1 and 4.1 ms.
__global__ __launch_bounds__(256, 7) void raygen_compat_sorted(GenArgs a)
{
    extern __shared__ __align__(16) float lds[];
    __shared__ __align__(16) uint32_t s_part[256];   // the slot's sequence; the scan's wave sums after
    const int nbin = a.nB * a.nQ;
    float* s_cdfb = lds;
    float* s_cdfg = s_cdfb + a.nB;                   // w / Ib of the drawn bins in (3)
    uint32_t* s_sob = (uint32_t*)(s_cdfg + nbin);
    int* s_ord = (int*)(s_sob + 64);
    uint32_t* s_hist = (uint32_t*)(s_ord + a.nB);    // w of the drawn bins in (3)
    uint32_t* s_cum = s_hist + nbin;
    const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63, wv = tid >> 6;
    for (int i = tid; i < a.nB; i += nth) {
        s_cdfb[i] = a.cdf_band[i];
        s_ord[i] = a.band_order[i];
    }
    for (int i = tid; i < nbin; i += nth) {
        s_cdfg[i] = a.cdf_g[i];
        s_hist[i] = 0u;
    }
    for (int i = tid; i < 64; i += nth) s_sob[i] = a.sobol_v[i];
    __syncthreads();
    const int R = a.rays_per_slot, L = a.run_len;
    const int h0 = tid * L < R ? tid * L : R;
    const int h1 = h0 + L < R ? h0 + L : R;
    const uint32_t xr0 = sobol_at(s_sob, lane), xr1 = sobol_at(s_sob + 32, lane);
    for (long long sl = blockIdx.x; sl < a.nslots; sl += gridDim.x) {
        const int4 si = a.slotinfo[a.slot0 + sl];
        const int cell = si.y;
        const int v = si.x % a.slots_per_emitter;
        const float Ti = a.T0[(size_t)a.snap * a.tstride0 + si.z];
        const long long q0 = sl * R;
        if (wv == 0) compat_sequence(a, cell, v, lane, s_part);
        __syncthreads();
        // (1) histogram of the (band, g) draws h0..h1-1
        if (h0 < h1) {
            Xorwow s = xorwow_jump(s_part, a.xw_poly + 5 * tid, a.xw_seed[5], (uint32_t)h0 * (uint32_t)a.draws_find);
            for (int h = h0; h < h1; ++h) {
                int band = cdf_search(s_cdfb, a.nB, u01_incl(xorwow_next(s)));
                int g = 0;
                if (a.g_search) g = cdf_search(s_cdfg + band * a.nQ, a.nQ, u01_incl(xorwow_next(s)));
                g = g > a.nQ - 1 ? a.nQ - 1 : g;
                atomicAdd(&s_hist[band * a.nQ + g], 1u);
            }
            if (!a.use_sobol) {   // the directions' 24-bit uniforms, taken up again in (3)
                s = xorwow_jump(s_part, a.xw_poly + 5 * (256 + tid), a.xw_seed[5],
                                (uint32_t)R * (uint32_t)a.draws_find + 2u * (uint32_t)h0);
                for (int h = h0; h < h1; ++h) {
                    a.w1[q0 + h] = xorwow_next(s) >> 8;
                    a.w0[q0 + h] = xorwow_next(s) >> 8;
                }
            }
        }
        __syncthreads();
        // (2) inclusive scan in replay order: entry k = p*nQ + g counts bin order[p]*nQ + g
        const int per = (nbin + nth - 1) / nth;
        const int k0 = tid * per < nbin ? tid * per : nbin;
        const int k1 = k0 + per < nbin ? k0 + per : nbin;
        const int p0 = (int)fdiv((uint32_t)k0, a.fd_nQ), g0 = k0 - p0 * a.nQ;
        uint32_t run = 0;
        for (int k = k0, p = p0, g = g0; k < k1; ++k) {
            run += s_hist[s_ord[p] * a.nQ + g];
            if (++g == a.nQ) { g = 0; ++p; }
        }
        uint32_t inc = run;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(inc, o);
            inc += lane >= o ? t : 0u;
        }
        if (lane == 63) s_part[wv] = inc;
        __syncthreads();
        inc -= run;
        for (int w = 0; w < wv; ++w) inc += s_part[w];
        for (int k = k0, p = p0, g = g0; k < k1; ++k) {
            const int band = s_ord[p], bin = band * a.nQ + g;
            const uint32_t cnt = s_hist[bin];
            inc += cnt;
            s_cum[k] = inc;
            if (cnt) {
                float w, winv, iib;
                bundle_weight(a, a.Ib, Ti, band, g, &w, &winv, &iib);
                s_hist[bin] = __float_as_uint(w);
                s_cdfg[bin] = winv;
            }
            if (++g == a.nQ) { g = 0; ++p; }
        }
        __syncthreads();
        // (3) bundles in chunks of 64 from n0 rounded down to a multiple of 64
        {
            const uint64_t n0 = (uint64_t)v * (uint64_t)R;
            const int lead = a.use_sobol ? (int)(n0 & 63ull) : 0;
            const int nch = (int)(((long long)lead + R + 63) / 64);
            const int c0 = (int)((long long)wv * nch / 4), c1 = (int)((long long)(wv + 1) * nch / 4);
            const int hf = max(64 * c0 - lead, 0);
            int lo = 0, hi = nbin - 1;             // first k with s_cum[k] > hf (s_cum[nbin-1] == R)
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (s_cum[mid] > (uint32_t)hf) hi = mid; else lo = mid + 1;
            }
            int kc = __builtin_amdgcn_readfirstlane(lo);
            uint64_t nb = n0 - (uint64_t)lead + 64ull * (uint64_t)c0;
            uint32_t x0 = sobol_at(s_sob, nb), x1 = sobol_at(s_sob + 32, nb);
            for (int c = c0; c < c1; ++c) {
                const int h = 64 * c - lead + lane, hl = min(64 * c - lead + 63, R - 1);
                int k = kc;                        // the first k with s_cum[k] > h
                for (bool more = true; more;) {
                    const int cl = (int)s_cum[min(kc + lane, nbin - 1)];
                    int i = 0;
                    for (; i < 64; ++i) {
                        const int ci = __builtin_amdgcn_readlane(cl, i);
                        if (ci > hl) break;
                        k += h >= ci ? 1 : 0;
                    }
                    more = i == 64;
                    kc += i;
                }
                const uint32_t mp = (x0 ^ xr0) >> 8, mt = (x1 ^ xr1) >> 8;
                if (h >= 0 && h < R) {
                    const long long q = q0 + h;
                    const int p = (int)fdiv((uint32_t)k, a.fd_nQ), g = k - p * a.nQ;
                    const int band = s_ord[p], bin = band * a.nQ + g;
                    uint32_t w0, w1;
                    if (a.use_sobol) desc_pack(mt, mp, band, g, &w0, &w1);
                    else desc_pack(a.w0[q], a.w1[q], band, g, &w0, &w1);
                    a.w0[q] = w0;
                    a.w1[q] = w1;
                    a.w[q] = __uint_as_float(s_hist[bin]);
                    a.winv[q] = s_cdfg[bin];
                }
                // Gray code of nb -> nb + 64: bits 5 and 6 + (trailing ones of nb / 64) change
                const int t = 6 + __builtin_ctzll(~(nb >> 6));
                x0 ^= s_sob[5] ^ (t < 32 ? s_sob[t] : 0u);
                x1 ^= s_sob[37] ^ (t < 32 ? s_sob[32 + t] : 0u);
                nb += 64;
            }
        }
        // the next slot's histogram and CDFs
        __syncthreads();
        for (int i = tid; i < nbin; i += nth) {
            s_hist[i] = 0u;
            s_cdfg[i] = a.cdf_g[i];
        }
    }
}

// -------------------------------------------------------------- trace ----
__device__ __forceinline__ gfloat* lev_T(const int* L)
{
    unsigned long long u = ((unsigned long long)(uint32_t)L[8] << 32) | (uint32_t)L[7];
    return (gfloat*)u;
}

// Temperature at a byte offset from the level base (a level of one snapshot
// stays within 4 GiB).
__device__ __forceinline__ float load_T(gfloat* base, int byte)
{
    typedef __attribute__((address_space(1))) const char gchar;
    return *(gfloat*)((gchar*)base + (uint32_t)byte);
}

// Smallest of three numbers (none NaN).
__device__ __forceinline__ float min3(float a, float b, float c)
{
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}


// Wave-aggregated tally atomics: the lanes with `need` set hand their running
// slot sums over, grouped by slot; each group is summed across the wave and
// its first lane adds the group total with three FP64 atomics.  Called by all
// 64 lanes (wave-uniform control flow).
__device__ __forceinline__ void flush_wave(const TraceArgs& P, bool need, int aslot, double aE, double aA,
                                           double aQ, int lane)
{
    unsigned long long m = __ballot(need);
    while (m) {
        const int leader = __ffsll((long long)m) - 1;
        const int s = __shfl(aslot, leader);
        const bool mine = need && aslot == s;
        double e = mine ? aE : 0.0, a = mine ? aA : 0.0, q = mine ? aQ : 0.0;
        for (int off = 32; off > 0; off >>= 1) {
            e += __shfl_xor(e, off);
            a += __shfl_xor(a, off);
            q += __shfl_xor(q, off);
        }
        if (lane == leader) {
            unsafeAtomicAdd(&P.E[s], e);
            unsafeAtomicAdd(&P.A[s], a);
            unsafeAtomicAdd(&P.Q2[s], q);
        }
        need = need && !mine;
        m = __ballot(need);
    }
}

// Tally one finished ray into the lane's running slot sums (TMODE 0; a lane
// whose sums belong to another slot has handed them over with flush_wave
// first) or the per-ray buffer (TMODE 1).
template <int TMODE>
__device__ __forceinline__ void tally_ray(const TraceArgs& P, float er, float ar, int rslot, uint32_t q, int& aslot,
                                          double& aE, double& aA, double& aQ)
{
    if (TMODE == 1) {
        P.pray[q] = make_float2(er, ar);
        return;
    }
    if (rslot != aslot) {
        aslot = rslot;
        aE = aA = aQ = 0.0;
    }
    const double de = (double)er, da = (double)ar, x = de - da;
    aE += de;
    aA += da;
    aQ += x * x;
}

// A drawn ray, as the refill hands it to a lane: packed (i, j, k) of the
// emitting cell, its tally slot, band | g << 16 | sign flags
// << 24, its processing slot in the launch, emitter temperature, direction and
// its reciprocals, weights, emission point (the cell centre).
struct RayStart {
    int cell, six, bg, ps;
    float Tc, sx, sy, sz, ix, iy, iz, rw, rwi, px, py, pz;
};

// Lane `src`'s ray (all 64 lanes call it).
__device__ __forceinline__ RayStart pull_ray(const RayStart& r, int src)
{
    RayStart o;
    o.cell = __shfl(r.cell, src);
    o.six = __shfl(r.six, src);
    o.bg = __shfl(r.bg, src);
    o.ps = __shfl(r.ps, src);
    o.Tc = __shfl(r.Tc, src);
    o.sx = __shfl(r.sx, src);
    o.sy = __shfl(r.sy, src);
    o.sz = __shfl(r.sz, src);
    o.ix = __shfl(r.ix, src);
    o.iy = __shfl(r.iy, src);
    o.iz = __shfl(r.iz, src);
    o.rw = __shfl(r.rw, src);
    o.rwi = __shfl(r.rwi, src);
    o.px = __shfl(r.px, src);
    o.py = __shfl(r.py, src);
    o.pz = __shfl(r.pz, src);
    return o;
}

// ------------------------------------------ learned draw inside the traversal
// The learned proposal of one emitting cell is evaluated by the whole wave
// whose queue draws that cell's rays: the network (features, two tanh
// layers, the output layer) and the running sums U of exp(clamp(z, -60, 60))
// over each head, written to the wave's row buffer in the layout of
// mlp_proposal's rows ([64 direction bins | nbin (band, g) bins | padding]).
// Each ray then searches the defensive mixture of both heads in that row
// (mix_search, as raygen_learned does from its rows).  It replaces, for the
// learned estimator, the draw from the fixed proposal that the reference
// makes where a bundle starts (code/mc_gpu.cu:138-144, find_band :830-896).
// Lane L computes columns col = 512 j + 8 L + c (j < 4, c < 8): the output
// layer's weights are then read 1 KB-contiguous per load instruction.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// c + a.lo b.lo + a.hi b.hi on BF16 pairs, FP32 accumulation (v_dot2_f32_bf16).
__device__ __forceinline__ float dot2bf(uint32_t a, uint32_t b, float c)
{
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}

__device__ __forceinline__ uint32_t readlane_u(uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); }

// A traversal kernel's argument block (its first argument, at offset 0 of the
// kernel argument segment) through a pointer the compiler cannot see through:
// fields read through it are loaded (scalar loads from the constant segment)
// where they are used instead of being hoisted to the kernel's start and held
// in scalar registers through the traversal loop.
typedef __attribute__((address_space(4))) const TraceArgs KArgs;
__device__ __forceinline__ KArgs* kernel_args()
{
    KArgs* k = (KArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return k;
}

// The row of emitting cell ijk (i | j << 10 | k << 20) of snapshot
// `snapshot` into U (all 64 lanes call it): H1 = tanh(X W1 + b1), H2 =
// tanh(H1 W2 + b2), Z = H2 W3 + b3, H1 and H2 rounded to BF16 as the training
// kernels round them, the products in FP32 from BF16 pairs; U per head from
// 8-column sums within a lane and exclusive lane scans across (the direction
// head is lanes 0..7 of chunk 0).
// An out-of-line call: the registers it needs are saved around the call,
// once per row, instead of pressing on the traversal loop's registers.
// Arguments are plain values (the network's pointers and sizes, the feature
// inputs), so the kernel's argument block stays in its constant segment.
__device__ __noinline__ void learned_row(const uint16_t* W1, const float* b1, const uint16_t* W2, const float* b2,
                                         const uint16_t* W3, const float* b3, int nbin, int noutp, const float* T0,
                                         int n0, int n1, int n2, int nbx, int nby, const float* centres, int co0,
                                         int co1, int co2, int bcp, int polar, float Lpolar, float inv_Tmax,
                                         float Tw_rel, int ijk, int lane, float* U)
{
    FeatArgs f;
    f.T0 = T0;
    f.n[0] = n0; f.n[1] = n1; f.n[2] = n2;
    f.nbx = nbx; f.nby = nby;
    f.centres = centres;
    f.coff[0] = co0; f.coff[1] = co1; f.coff[2] = co2;
    f.bc_periodic = bcp;
    f.polar = polar;
    f.Lpolar = Lpolar;
    f.inv_Tmax = inv_Tmax;
    f.Tw_rel = Tw_rel;
    float x[kMlpIn];
    cell_features(f, ijk & 1023, (ijk >> 10) & 1023, (ijk >> 20) & 1023, x);
    MlpWeights w;
    w.W1 = W1; w.b1 = b1; w.W2 = W2; w.b2 = b2; w.W3 = W3; w.b3 = b3;
    w.nbin = nbin; w.noutp = noutp;
    w.W2T = nullptr; w.W3T = nullptr;
    float a1 = w.b1[lane];
#pragma unroll
    for (int i = 0; i < kMlpIn; ++i) a1 = fmaf(x[i], bf2f(w.W1[i * kMlpHid + lane]), a1);
    const uint32_t h1 = f2bf(tanhf(a1));
    float a2 = w.b2[lane];
    for (int kp = 0; kp < kMlpHid / 2; ++kp) {
        const uint32_t hp = readlane_u(h1, 2 * kp) | (readlane_u(h1, 2 * kp + 1) << 16);
        const uint32_t wp = (uint32_t)w.W2[(2 * kp) * kMlpHid + lane] | ((uint32_t)w.W2[(2 * kp + 1) * kMlpHid + lane] << 16);
        a2 = dot2bf(hp, wp, a2);
    }
    const uint32_t h2 = f2bf(tanhf(a2));
    const int nout = kMlpDir + w.nbin;
    float base = 0.f;   // the (band, g) head's sum over the previous chunks
    for (int j = 0; j < 4; ++j) {
        const int col = 512 * j + 8 * lane;
        float a[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) a[c] = 0.f;
        if (col < noutp) {
            const uint16_t* r = w.W3 + col;
#pragma unroll 2
            for (int kp = 0; kp < kMlpHid / 2; ++kp) {
                const uint32_t hp = readlane_u(h2, 2 * kp) | (readlane_u(h2, 2 * kp + 1) << 16);
                const uint4 u0 = *(const uint4*)(r + (size_t)(2 * kp) * noutp);
                const uint4 u1 = *(const uint4*)(r + (size_t)(2 * kp + 1) * noutp);
                a[0] = dot2bf(hp, __builtin_amdgcn_perm(u1.x, u0.x, 0x05040100u), a[0]);
                a[1] = dot2bf(hp, __builtin_amdgcn_perm(u1.x, u0.x, 0x07060302u), a[1]);
                a[2] = dot2bf(hp, __builtin_amdgcn_perm(u1.y, u0.y, 0x05040100u), a[2]);
                a[3] = dot2bf(hp, __builtin_amdgcn_perm(u1.y, u0.y, 0x07060302u), a[3]);
                a[4] = dot2bf(hp, __builtin_amdgcn_perm(u1.z, u0.z, 0x05040100u), a[4]);
                a[5] = dot2bf(hp, __builtin_amdgcn_perm(u1.z, u0.z, 0x07060302u), a[5]);
                a[6] = dot2bf(hp, __builtin_amdgcn_perm(u1.w, u0.w, 0x05040100u), a[6]);
                a[7] = dot2bf(hp, __builtin_amdgcn_perm(u1.w, u0.w, 0x07060302u), a[7]);
            }
        }
        // e = exp(clamp(z)), running sums within the lane's 8 columns
        float run = 0.f;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (col + c < nout) run += __expf(fminf(fmaxf(a[c] + w.b3[col + c], -60.f), 60.f));
            a[c] = run;
        }
        // exclusive scan of the lanes' sums, the direction head on its own
        const int seg = (j == 0 && lane >= 8) ? 8 : 0;
        float incl = run;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float t = __shfl_up(incl, o);
            if (lane - o >= seg) incl += t;
        }
        float excl = __shfl_up(incl, 1);
        if (lane == seg) excl = 0.f;
        const float sb = (j == 0 && lane < 8) ? excl : base + excl;
        if (col < noutp) {
            float4* d = (float4*)(U + col);
            d[0] = make_float4(sb + a[0], sb + a[1], sb + a[2], sb + a[3]);
            d[1] = make_float4(sb + a[4], sb + a[5], sb + a[6], sb + a[7]);
        }
        base = base + __shfl(incl, 63);
    }
}

// Whether ray q of snapshot qs of a fused launch, with polar uniform bits mt
// (m_theta of the plain draw), is a listed long-ray candidate
// (TraceArgs::cand): one integer test for cand_scan and the traversal's draw.
template <typename A>
__device__ __forceinline__ bool long_candidate(const A& P, uint32_t q, uint32_t qs, uint32_t mt)
{
    FastDiv fd;   // (field by field: P may be the kernel argument segment)
    fd.m = P.cand_fd.m;
    fd.s = P.cand_fd.s;
    fd.d = P.cand_fd.d;
    const uint32_t x = fdiv(q, fd);
    return qs + 1u == (uint32_t)P.nsnap_launch && q - x * fd.d >= P.cand_from &&
           mt - (1u << 23) + P.cand_w < 2u * P.cand_w;
}

// Crossings per iteration of the traversal, their field loads in flight together
// (a wave's lanes meet an L2 miss nearly every crossing, and only four waves
// per SIMD hide it).  A ray that ends inside an iteration wastes the rest.
// 384x256x256 on one level: 403 / 371 / 378 / 386 / 398 ms at 1 / 2 / 3 / 4 / 6
// (the loop before: 398; L2 reads per crossing 0.88 -> 0.64, VALU instructions
// 2.19 -> 1.76); two coarsened 256x128x128 snapshots, five crossings on each
// finer level: 48.0 / 47.3 / 45.6 / 49.0 / 42.8 ms at 1 / 2 / 3 / 4 / 5 (44.4).
constexpr int kAheadFine = 2, kAheadLev = 5;
constexpr int kQuads = 16;   // rays a wave follows in the drain, four lanes each
constexpr int kDrain = 16;   // crossings a ray moves ahead per batch of the drain (a multiple of 4)

// Value of another lane of the quad (4 consecutive lanes): lane j of the quad
// reads lane (CTRL >> 2 j) & 3.
template <int CTRL>
__device__ __forceinline__ int quad_i(int v)
{
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float quad_f(float v)
{
    return __int_as_float(quad_i<CTRL>(__float_as_int(v)));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kQuadPrev = 0x93;
// Minimum over the quad (no NaN): v_min_f32 with the permuted operand; s_nop 1
// gives the two wait states between a VALU write and its DPP read.
__device__ __forceinline__ float quad_min(float v)
{
    float r;
    asm("s_nop 1\n\tv_min_f32_dpp %0, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_min_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
        : "=&v"(r)
        : "v"(v));
    return r;
}
// acc = fma(x of lane j of the quad, y_j, acc) for j = 0..3 in turn (s_nop 1:
// the two wait states before the first DPP read of x); t: acc after each.
#define DN_QFMA(x, y, j) "v_fmac_f32_dpp %0, " x ", " y " quad_perm:[" j "," j "," j "," j "] row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void quad_fma(float& acc, float x, float y0, float y1, float y2, float y3)
{
    asm("s_nop 1\n\t" DN_QFMA("%1", "%2", "0") DN_QFMA("%1", "%3", "1") DN_QFMA("%1", "%4", "2") DN_QFMA("%1", "%5", "3")
        : "+&v"(acc)
        : "v"(x), "v"(y0), "v"(y1), "v"(y2), "v"(y3));
}
__device__ __forceinline__ void quad_fma_t(float& acc, float x, const float* y, float* t)
{
    asm("s_nop 1\n\t" DN_QFMA("%4", "%5", "0") "v_mov_b32 %1, %0\n\t" DN_QFMA("%4", "%6", "1") "v_mov_b32 %2, %0\n\t"
        DN_QFMA("%4", "%7", "2") "v_mov_b32 %3, %0\n\t" DN_QFMA("%4", "%8", "3")
        : "+&v"(acc), "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2])
        : "v"(x), "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]));
    t[3] = acc;
}
__device__ __forceinline__ int quad_sum(int v)
{
    v += quad_i<kQuadXor1>(v);
    return v + quad_i<kQuadXor2>(v);
}
template <int CTRL>
__device__ __forceinline__ double quad_d(double v)
{
    const int2 u = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(double, make_int2(quad_i<CTRL>(u.x), quad_i<CTRL>(u.y)));
}
// Lane a of a quad: the quad's sum of v[a].
__device__ __forceinline__ int quad_spread(const int* v, int a)
{
    const bool odd = a & 1, hi = a & 2;
    const int p = (odd ? v[1] : v[0]) + quad_i<kQuadXor1>(odd ? v[0] : v[1]);
    const int q = (odd ? v[3] : v[2]) + quad_i<kQuadXor1>(odd ? v[2] : v[3]);
    return (hi ? q : p) + quad_i<kQuadXor2>(hi ? p : q);
}
__device__ __forceinline__ int quad_max(int v)
{
    v = max(v, quad_i<kQuadXor1>(v));
    return max(v, quad_i<kQuadXor2>(v));
}
__device__ __forceinline__ int quad_min_i(int v)
{
    v = min(v, quad_i<kQuadXor1>(v));
    return min(v, quad_i<kQuadXor2>(v));
}

// The long-ray candidates of a fused launch: each ray of the final part of
// the 8 XCD ranges of the launch's last snapshot (nfin rays per range from
// cand_from on, those below nrays) gets the plain draw's Philox block, and
// the rays that pass long_candidate go to their range's list (list x at
// x * cand_cap, its count at cand_cnt[64 x]; every hit is counted, also past
// cand_cap).  A block takes tiles of kCandTile rays of one range and stages
// the tile's hits in LDS: one global atomic per tile.
constexpr uint32_t kCandTile = 4096;
__global__ __launch_bounds__(256) void cand_scan(TraceArgs P, uint32_t nfin, uint32_t* list)
{
    __shared__ uint32_t s_q[kCandTile];
    __shared__ uint32_t s_n, s_base;
    const uint32_t qs = (uint32_t)P.nsnap_launch - 1u;
    const uint32_t tpr = (nfin + kCandTile - 1u) / kCandTile;   // tiles per range
    for (uint32_t t = blockIdx.x; t < 8u * tpr; t += gridDim.x) {
        const uint32_t x = t / tpr;
        const uint32_t j0 = (t - x * tpr) * kCandTile;
        const uint32_t jn = min(kCandTile, nfin - j0);
        const uint32_t q0 = x * P.cand_fd.d + P.cand_from + j0;
        if (threadIdx.x == 0) s_n = 0u;
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < jn; j += blockDim.x) {
            const uint32_t q = q0 + j;
            if (q < (uint32_t)P.nrays) {
                const uint32_t slot = fdiv(q, P.fd_R);
                const uint32_t r = q - slot * (uint32_t)P.rays_per_slot;
                const int4 si = P.slotinfo[P.slot0 + slot];
                const u32x4 h = philox4x32_10(u32x4{r, (uint32_t)si.y, (uint32_t)(P.snap + (int)qs), 0u},
                                              (uint32_t)P.seed, (uint32_t)(P.seed >> 32));
                if (long_candidate(P, q, qs, h.z >> 8)) s_q[atomicAdd(&s_n, 1u)] = q;
            }
        }
        __syncthreads();
        const uint32_t n = s_n;
        if (threadIdx.x == 0 && n) s_base = atomicAdd(P.cand_cnt + 64u * x, n);
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < n; k += blockDim.x)
            if (s_base + k < P.cand_cap) list[(size_t)x * P.cand_cap + s_base + k] = s_q[k];
        __syncthreads();   // the tile's hits are out before the next tile's reset
    }
}

// Persistent cell-by-cell traversal (code/mc_gpu.cu:228-438).
//
// Work: the launch's rays (in 3-D brick order of their emitting cells) are
// cut into super-chunks of `super` consecutive rays.  Blocks are dispatched
// round-robin over the 8 XCDs, so XCD x owns the contiguous super-chunk range
// [x*N/8, (x+1)*N/8); its waves claim super-chunks of that range in order from
// a per-XCD counter (one atomic per super-chunk), so the rays in flight on an
// XCD stay inside a compact region its L2 holds and the 64 lanes of a wave
// trace consecutive rays of the same one to three cells.  A wave whose XCD
// range is used up claims from the next XCD's range, so no XCD idles while
// another still has work.  The grid is sized to the resident capacity.
//
// Lanes whose ray ended stay idle until `refill_k` lanes of the wave are idle
// (or none is alive); one wave-uniform refill block then tallies the finished
// rays and starts new rays on every idle lane, in lane order.  With atomic
// tallies and no records (QUEUE) the new rays come from the wave's queue of 64
// drawn rays (lane j holds ray gbase + j), redrawn 64 at a time on the whole
// wave; otherwise each idle lane draws its own ray.
//
// Tallies: QUEUE keeps a ring of kRing slot accumulators per wave in LDS
// (FP64 E, A, sum x^2): the processing slots of a drawn queue get entries
// (slot mod kRing; an entry still holding an older slot first adds its sums
// to that slot with three device FP64 atomics), and a finished ray adds to
// its entry with LDS atomics while the entry holds its slot, else straight to
// the slot.  TMODE 0 with records keeps a running FP64 sum per lane, handed
// over with wave-aggregated atomics (flush_wave) when the lane moves to
// another slot.  TMODE 1 writes each ray's (E, A) for the deterministic
// reduce_rays pass.
//
// One iteration: a lane first walks kAhead crossings (distances, face snap,
// move, boundary; which cells a ray crosses does not depend on the field) with
// each next cell's field load issued as its offsets are known, then the table
// lookups, optical depth, transmissivity and gathered emission of the same
// crossings follow in order, each taking the field value of the crossing
// before.  With the kappa/Ib slice in LDS the field holds table coordinates
// (t_to_u).  A wave's last rays are followed by four lanes each (the drain).
//
// GEN: the rays are drawn in the kernel instead of read from descriptors
// (1: the plain estimator's Philox draw, bit-identical to raygen_plain; 2:
// the learned proposal, evaluated per emitting cell by the wave that draws
// its rays, see learned_row), and one launch covers every snapshot: XCD x's
// claims walk snapshot by snapshot through its 1/8 of each snapshot's
// super-chunks, so all XCDs work on the same snapshot at a time.
//
// Long rays first (GEN == 1, a list from cand_scan): a ray along the walls
// of an optically thin bin can run to the step cap, tens of ms on its own;
// started among the launch's last rays it would hold the launch open after
// all other work is done.  The waves draw their queues from the list first
// and skip the listed rays (the same test) where their super-chunks come up:
// every ray is still traced once, with the same arithmetic.
template <int SPEC, int TAB, int TMODE, bool REC, bool AMC, int GEN>
__global__ __launch_bounds__(TAB == kTabSliced ? 1024 : 256) void trace(TraceArgs P)
{
    extern __shared__ float lds[];
    // the wave's tally ring (atomic tallies, no records), first in LDS:
    // kRing entries of FP64 (E, A, sum x^2), the processing slot each holds
    // (-1: free) and its tally slot
    constexpr bool QUEUE = TMODE == 0 && !REC;
    const int nwv = QUEUE ? (int)(blockDim.x >> 6) : 0;
    const int rb = (int)(threadIdx.x >> 6) * kRing;   // this wave's first entry
    double* s_rv = (double*)lds;
    int* s_rt = (int*)(s_rv + 3 * kRing * nwv);
    int* s_rg = s_rt + kRing * nwv;
    int* s_lev = s_rg + kRing * nwv;            // 6 * kLevWords
    float* s_face = (float*)(s_lev + 6 * kLevWords);
    int* s_off = (int*)(s_face + P.nfaces);     // brick offsets per level and axis
    float* s_ibw = (float*)(s_off + P.noffs);   // 6 * nB wall Planck values
    // words of LDS by address (an address is one register, no base to add)
    typedef __attribute__((address_space(3))) const float lfloat;
    typedef __attribute__((address_space(3))) const int lint;
    auto lds_at = [&](const void* q) -> int { return (int)(uint32_t)(uintptr_t)(lfloat*)q; };
    auto lds_f = [&](int at) -> float { return *(lfloat*)(uintptr_t)(uint32_t)at; };
    auto lds_i = [&](int at) -> int { return *(lint*)(uintptr_t)(uint32_t)at; };
    const int face0 = lds_at(s_face), off0 = lds_at(s_off);
    float* s_ib = s_ibw + 6 * P.nB;             // Ib rows (nT or tab_nw nodes)
    const int nw = P.tab_nw;
    float* s_kq = s_ib + P.nB * nw;             // sliced kappa rows (kTabSliced)
    // GEN: band CDF after the tables that are in LDS
    float* s_cdfb = TAB == kTabSliced ? s_kq + P.nB * P.nQ * nw : (TAB == kTabIbLds ? s_ib + P.nB * P.nT : s_ib);
    float* s_cdfg = s_cdfb + P.nB;              // GEN, gen_lds bit 0: g CDF rows; bit 1: 1/(k Ib)(Tmax)
    float* s_iem = s_cdfg + P.nB * P.nQ;
    for (int i = threadIdx.x; i < P.nlev; i += blockDim.x) {
        int* L = s_lev + i * kLevWords;
        L[0] = P.lev[i].n[0]; L[1] = P.lev[i].n[1]; L[2] = P.lev[i].n[2];
        // per axis: LDS address of face 0
        L[3] = face0 + 4 * P.lev[i].foff[0]; L[4] = face0 + 4 * P.lev[i].foff[1]; L[5] = face0 + 4 * P.lev[i].foff[2];
        L[6] = P.lev[i].maxs;
        const float* tb = P.T[i] + (size_t)P.snap * P.lev[i].tstride;
        unsigned long long u = (unsigned long long)tb;
        L[7] = (int)(uint32_t)u;
        L[8] = (int)(uint32_t)(u >> 32);
        // from a cell's low face (word c - 1 of 1-based cell c) to its word of the
        // brick-offset table
        for (int a = 0; a < 3; ++a) L[11 + a] = off0 - face0 + 4 * (P.lev[i].ooff[a] - P.lev[i].foff[a]);
        L[14] = (int)P.lev[i].tstride;
        int before = 0;                          // crossings on the finer levels
        for (int g = 0; g < i; ++g) before += P.lev[g].maxs;
        L[15] = before;
    }
    for (int i = threadIdx.x; i < P.nfaces; i += blockDim.x) s_face[i] = P.faces[i];
    for (int i = threadIdx.x; i < P.noffs; i += blockDim.x) s_off[i] = P.offs[i];
    for (int i = threadIdx.x; i < 6 * P.nB; i += blockDim.x) s_ibw[i] = P.Ibw[i];
    if (QUEUE && (threadIdx.x & 63) < kRing) {
        const int e = rb + (int)(threadIdx.x & 63);
        s_rt[e] = -1;
        s_rg[e] = 0;
        s_rv[3 * e] = s_rv[3 * e + 1] = s_rv[3 * e + 2] = 0.0;
    }
    if (GEN) {
        for (int i = threadIdx.x; i < P.nB; i += blockDim.x) s_cdfb[i] = P.cdf_band[i];
        if (P.gen_lds & 1)
            for (int i = threadIdx.x; i < P.nB * P.nQ; i += blockDim.x) s_cdfg[i] = P.cdf_g[i];
        if (P.gen_lds & 2)
            for (int i = threadIdx.x; i < P.nB * P.nQ; i += blockDim.x) s_iem[i] = P.inv_emax[i];
    }
    if (SPEC == kSpecTable && TAB == kTabIbLds)
        for (int i = threadIdx.x; i < P.nB * P.nT; i += blockDim.x) s_ib[i] = P.Ib[i];
    if (SPEC == kSpecTable && TAB == kTabSliced) {
        // (a slice that reaches the table's top may end with its last node again)
        for (int i = threadIdx.x; i < P.nB * nw; i += blockDim.x) {
            const int r = i / nw;
            s_ib[i] = P.Ib[r * P.nT + min(P.tab_lo + (i - r * nw), P.nT - 1)];
        }
        for (int i = threadIdx.x; i < P.nB * P.nQ * nw; i += blockDim.x) {
            const int r = i / nw;
            s_kq[i] = P.kq[r * P.nT + min(P.tab_lo + (i - r * nw), P.nT - 1)];
        }
    }
    __syncthreads();
    const float* ibt = TAB == kTabGlobal ? P.Ib : s_ib;
    gfloat* kq = (gfloat*)P.kq;
    const int rowlen = TAB == kTabSliced ? nw : P.nT;   // nodes per table row
    // a ray's table rows: element indices, or (sliced) LDS word indices
    const int kr0 = TAB == kTabSliced ? lds_at(s_kq) >> 2 : 0;
    const int ir0 = TAB == kTabSliced ? lds_at(s_ib) >> 2 : 0;

    const int lane = threadIdx.x & 63;
    const unsigned nb = gridDim.x, b = blockIdx.x;
    const uint32_t nrays = (uint32_t)P.nrays;   // rays per snapshot of the launch
    const uint32_t S = (uint32_t)P.super;
    const uint32_t cps = (nrays + S - 1) / S;   // super-chunks per snapshot
    const bool split = (nb % 8u) == 0u;
    const uint32_t xcd = split ? b % 8u : 0u;
    const uint32_t nparts = split ? 8u : 1u;
    const uint32_t per_x = (cps + nparts - 1u) / nparts;        // per XCD and snapshot
    const uint32_t nclaim = per_x * (uint32_t)P.nsnap_launch;   // claims of one XCD counter
    const int nT = P.nT;

    // wave-uniform cursor over the claimed super-chunk (rays cur..cend of snapshot csnap)
    uint32_t xi = 0, cur = 0, cend = 0, csnap = 0;
    bool more = true;
    // lane state
    bool alive = false, fin = false;
    uint32_t qcur = 0;
    int rslot = -1, aslot = -1;
    double aE = 0.0, aA = 0.0, aQ = 0.0;
    uint32_t steps_lane = 0;
    int endt = 0;
    float Dfin = 1.0f;
    float px = 0.f, py = 0.f, pz = 0.f, sx = 1.f, sy = 1.f, sz = 1.f, ix = 1.f, iy = 1.f, iz = 1.f;
    float fx = 0.f, fy = 0.f, fz = 0.f, tau = 0.f, tra = 1.f, G = 0.f, rw = 0.f, rwi = 0.f, Tc = 0.f;
    // The ray's cell, as three LDS addresses: A_a of its exit face along axis a
    // (bytes; + s_a, +-4, one cell further), and A_a + K_a its word of the
    // axis's brick-offset table.
    int A0 = s_lev[3], A1 = s_lev[4], A2 = s_lev[5], K0 = s_lev[11], K1 = s_lev[12], K2 = s_lev[13];
    int s0 = 4, s1 = 4, s2 = 4;
    int krow = 0, ibrow = 0, band = 0, lev = 0, cnt = 0, rsteps = 0;
    uint32_t hash = 2166136261u;
    int maxs = s_lev[6];
    if (!AMC) maxs = __builtin_amdgcn_readfirstlane(maxs);
    // level 0's LDS addresses (scalar registers: every ray starts there)
    const int f00 = __builtin_amdgcn_readfirstlane(s_lev[3]), f01 = __builtin_amdgcn_readfirstlane(s_lev[4]);
    const int f02 = __builtin_amdgcn_readfirstlane(s_lev[5]), k00 = __builtin_amdgcn_readfirstlane(s_lev[11]);
    const int k01 = __builtin_amdgcn_readfirstlane(s_lev[12]), k02 = __builtin_amdgcn_readfirstlane(s_lev[13]);
    // 0-based cell along axis a of the level block L
    auto cell_of = [&](const int* L, int a, int A, int s) -> int { return ((A - L[3 + a]) >> 2) - (s > 0 ? 1 : 0); };
    gfloat* Tl = lev_T(s_lev);
    gfloat* T0 = Tl;
    uint32_t rsnap = 0;
    // the wave's queue of drawn rays (lane j: ray gbase + j, j < gn); the
    // per-ray outputs (TMODE 1) and records index rays by lane, so they keep
    // the direct hand-out
    uint32_t gn = 0, ghead = 0, gsnap = 0;
    int pslot = 0;                        // processing slot of the lane's ray (tally ring tag)
    const int nslot_l = (int)(nrays / (uint32_t)P.rays_per_slot);   // processing slots per snapshot
    // the finished ray's (e, a): into its ring entry while the entry holds its
    // slot, else (evicted) straight to the tally
    auto ring_tally = [&](float er, float ar) {
        const double de = (double)er, da = (double)ar, x = de - da;
        const int e = rb + (pslot & (kRing - 1));
        if (s_rt[e] == pslot) {
            __hip_atomic_fetch_add(&s_rv[3 * e], de, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(&s_rv[3 * e + 1], da, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(&s_rv[3 * e + 2], x * x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
            unsafeAtomicAdd(&P.E[rslot], de);
            unsafeAtomicAdd(&P.A[rslot], da);
            unsafeAtomicAdd(&P.Q2[rslot], x * x);
        }
    };
    // The finished rays of all lanes.  Where they share one slot and its ring
    // entry, the sum of each 16 lanes is added once: the atomics of lanes on one
    // address take the LDS one lane after the other.  For descriptor launches of
    // at least 256 rays per slot, where most refills meet one slot.  Traversal of
    // reference sampling without and with it, by rays per slot (three levels,
    // sorted bands): 100 10.3 / 10.3 ms, 160 11.7 / 11.7, 256 19.5 / 18.9, 800
    // 7.33 / 7.03, 5000 34.0 / 31.0, 20000 (2.6 crossings) 12.4 / 10.7 (quads: 10.9);
    // learned rays on four levels: 100 and 160 the same, 256 4.79 / 4.63, 400 7.70 /
    // 7.26, 1600 27.4 / 25.1; on one level the same within 1 % up to 1600.  A fused
    // launch of 500 per slot is no faster.
    const bool wide = QUEUE && GEN == 0 && P.rays_per_slot >= 256;
    auto ring_tally_wave = [&](bool f, float er, float ar) {
        const unsigned long long fm = __ballot(f);
        if (!fm) return;
        const int p0 = __builtin_amdgcn_readlane(pslot, __builtin_ctzll(fm));
        const int e0 = rb + (p0 & (kRing - 1));
        if (__ballot(f && pslot != p0) == 0ull && s_rt[e0] == p0) {
            double de = f ? (double)er : 0.0, da = f ? (double)ar : 0.0;
            double q = (de - da) * (de - da);
            de += quad_d<kQuadXor1>(de);
            da += quad_d<kQuadXor1>(da);
            q += quad_d<kQuadXor1>(q);
            de += quad_d<kQuadXor2>(de);
            da += quad_d<kQuadXor2>(da);
            q += quad_d<kQuadXor2>(q);
            de += quad_d<0x141>(de);
            da += quad_d<0x141>(da);
            q += quad_d<0x141>(q);
            de += quad_d<0x140>(de);
            da += quad_d<0x140>(da);
            q += quad_d<0x140>(q);
            if ((lane & 15) == 0 && ((fm >> lane) & 0xFFFFull)) {
                __hip_atomic_fetch_add(&s_rv[3 * e0], de, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(&s_rv[3 * e0 + 1], da, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(&s_rv[3 * e0 + 2], q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        } else if (f) {
            ring_tally(er, ar);
        }
    };
    // ring entry e's sums to its tally slot (one lane)
    auto ring_flush = [&](int e) {
        const int t = s_rg[e];
        unsafeAtomicAdd(&P.E[t], s_rv[3 * e]);
        unsafeAtomicAdd(&P.A[t], s_rv[3 * e + 1]);
        unsafeAtomicAdd(&P.Q2[t], s_rv[3 * e + 2]);
    };
    RayStart Qr = {};
    // learned draw (GEN == 2): this lane's drawn bins and p/q for draw_ray, and
    // the wave's cached proposal row (processing slot and snapshot)
    int lr_band = 0, lr_g = 0;
    uint32_t lr_mt = 0, lr_mp = 0;
    float lr_ratio = 0.f;
    uint32_t row_slot = 0xFFFFFFFFu, row_snap = 0xFFFFFFFFu;
    const uint32_t wave_id = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    // long rays first, one scalar: bit 8 on (off when a list found more rays
    // than it holds; with none found no ray passes the test either), bit 31
    // while the wave still draws from the lists, bits 0..3 the lists it has
    // used up (its XCD's first, then the following XCDs')
    uint32_t cand = 0;
    if (GEN == 1 && QUEUE && P.cand != nullptr) {
        uint32_t tot = 0;
        bool fits = true;
        for (int x = 0; x < 8; ++x) {
            const uint32_t n = __builtin_amdgcn_readfirstlane(P.cand_cnt[64 * x]);
            fits = fits && n <= P.cand_cap;
            tot += n;
        }
        cand = fits && tot > 0u ? 0x80000100u : 0u;
    }

    // ray q of snapshot qs of the launch: drawn here (GEN, the plain estimator's
    // Philox draw, bit-identical to raygen_plain) or read from its descriptors.
    // A listed long ray drawn from its super-chunk (not from the list) comes
    // back with bit 31 of bg set: it is not started there.
    auto draw_ray = [&](uint32_t q, uint32_t qs, bool listed) -> RayStart {
        RayStart rd;
        const uint32_t slot = fdiv(q, P.fd_R);
        const int4 si = P.slotinfo[P.slot0 + slot];
        rd.six = si.x;
        rd.cell = si.w;
        rd.ps = (int)slot + (int)qs * nslot_l;
        rd.px = P.centres[P.coff[0] + (si.w & 1023) + 1];
        rd.py = P.centres[P.coff[1] + ((si.w >> 10) & 1023) + 1];
        rd.pz = P.centres[P.coff[2] + ((si.w >> 20) & 1023) + 1];
        gfloat* Te = lev_T(s_lev) + (GEN ? (size_t)qs * (uint32_t)s_lev[14] : (size_t)0);
        const float Tq = Te[si.z];
        rd.Tc = Tq;
        int bnd, g;
        uint32_t mt, mp;
        float ratio = 1.0f;       // p/q of a learned descriptor
        bool weigh = GEN;         // emission weight computed here (tables in LDS)
        bool skip = false;        // a listed long ray, traced from the list
        if (GEN == 1) {
            const uint32_t r = q - slot * (uint32_t)P.rays_per_slot;
            const u32x4 x = philox4x32_10(u32x4{r, (uint32_t)si.y, (uint32_t)(P.snap + (int)qs), 0u},
                                          (uint32_t)P.seed, (uint32_t)(P.seed >> 32));
            bnd = cdf_search(s_cdfb, P.nB, u01_open(x.x));
            if (!P.g_search)
                g = 0;
            else if (P.gen_lds & 1)
                g = cdf_search(s_cdfg + bnd * P.nQ, P.nQ, u01_open(x.y));
            else
                g = cdf_search(P.cdf_g + bnd * P.nQ, P.nQ, u01_open(x.y));
            g = g > P.nQ - 1 ? P.nQ - 1 : g;
            mt = x.z >> 8;
            mp = x.w >> 8;
            // (the test's arguments read from the kernel argument segment here)
            skip = (cand & 0x100u) && !listed && long_candidate(*kernel_args(), q, qs, mt);
        } else if (GEN == 2) {
            bnd = lr_band;
            g = lr_g;
            mt = lr_mt;
            mp = lr_mp;
            ratio = lr_ratio;
        } else {
            const uint32_t a0 = P.w0[q], a1 = P.w1[q];
            bnd = desc_band(a0, a1);
            g = desc_g(a1);
            mt = a0 & 0xFFFFFFu;
            mp = a1 & 0xFFFFFFu;
            if (P.desc_ratio) {
                ratio = P.w[q];
                weigh = true;
            } else {
                rd.rw = P.w[q];
                rd.rwi = P.winv[q];
            }
        }
        if (weigh) {
            // Ibmax (k_i Ib_i) / (k_max Ib_max) (code/mc_gpu.cu:63, :163-169),
            // the arithmetic of the generators' bundle weights
            float kap, ib;
            if (SPEC == kSpecGreyT4) {
                const float t2 = Tq * Tq;
                kap = P.kappa_grey;
                ib = t2 * t2;
            } else {
                // sliced tables: Tq is the table coordinate within the slice
                int t;
                float fr;
                if (TAB == kTabSliced) {
                    t = (int)Tq;
                    t = t > nw - 2 ? nw - 2 : t;
                    fr = Tq - (float)t;
                } else {
                    float pos = fmaf(Tq, P.inv_dT, P.mT0);
                    pos = fminf(fmaxf(pos, 0.0f), (float)(nT - 1));
                    t = (int)pos;
                    t = t > nT - 2 ? nT - 2 : t;
                    fr = pos - (float)t;
                }
                const int kr = (bnd * P.nQ + g) * rowlen, ir = bnd * rowlen;
                const float k0 = TAB == kTabSliced ? s_kq[kr + t] : kq[kr + t];
                const float k1 = TAB == kTabSliced ? s_kq[kr + t + 1] : kq[kr + t + 1];
                const float i0 = ibt[ir + t], i1 = ibt[ir + t + 1];
                kap = fmaf(fr, k1 - k0, k0);
                ib = fmaf(fr, i1 - i0, i0);
            }
            const float iem = (P.gen_lds & 2) ? s_iem[bnd * P.nQ + g] : P.inv_emax[bnd * P.nQ + g];
            const float w = P.Ibmax * (kap * ib) * iem;
            const float wi = w * (1.0f / ib);
            rd.rw = GEN == 1 ? w : w * ratio;
            rd.rwi = GEN == 1 ? wi : wi * ratio;
        }
        const float ut = ((float)mt + P.u_off) * kTwoM24;
        const float up = ((float)mp + P.u_off) * kTwoM24;
        const float cth = 1.0f - 2.0f * ut;
        const float sth = 2.0f * sqrtf(ut * (1.0f - ut));
        float sp, cp;
        sincos2pi(up, &sp, &cp);
        const float s1 = sth * cp, s2 = sth * sp;
        float dx = P.polar == 0 ? cth : (P.polar == 1 ? s2 : s1);
        float dy = P.polar == 0 ? s1 : (P.polar == 1 ? cth : s2);
        float dz = P.polar == 0 ? s2 : (P.polar == 1 ? s1 : cth);
        if (dx == 0.0f) dx = 1e-10f;
        if (dy == 0.0f) dy = 1e-10f;
        if (dz == 0.0f) dz = 1e-10f;
        const int f = (dx < 0.0f ? 1 : 0) | (dy < 0.0f ? 2 : 0) | (dz < 0.0f ? 4 : 0);
        rd.sx = dx; rd.sy = dy; rd.sz = dz;
        rd.ix = 1.0f / dx;
        rd.iy = 1.0f / dy;
        rd.iz = 1.0f / dz;
        rd.bg = bnd | (g << 16) | (f << 24) | (skip ? (int)(1u << 31) : 0);
        return rd;
    };

    // Next claim of XCD X's share (nclaim or more: none left).  Another XCD's
    // counter is read first: in a small launch every wave visits all eight at
    // the end, and reads of a used-up counter do not queue as atomics do.
    auto claim_of = [&](uint32_t X) -> uint32_t {
        uint32_t c = 0;
        if (lane == 0) {
            if (xi > 0u) c = __hip_atomic_load(P.claim + 32u * X, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (c < nclaim) c = atomicAdd(P.claim + 32u * X, 1u);
        }
        return __builtin_amdgcn_readfirstlane(c);
    };
    // Retiring: a wave asked to claim more work near the launch's end (its last
    // claim at retire_from or later) while one of its rays is beyond ask_at
    // crossings stops claiming, so that it reaches the drain below (105 ns per
    // crossing against some 850 at the bulk's pace) while the other waves trace
    // the rest.  At most
    // retire_most waves of the launch do for rays beyond retire_steps (counted
    // in claim word 16), as many beyond twice that for the waves that were
    // refused (word 17), and so on up to word 19: the longest rays are not left
    // out, and the other waves remain to claim what is left.
    uint32_t last_c = 0, asked = 0;
    int ask_at = P.retire_most > 0u ? P.retire_steps : 0x7FFFFFFF;
    auto retire = [&]() -> bool {
        if (last_c < P.retire_from || !__ballot(alive && cnt > ask_at)) return false;
        uint32_t k = 0;
        if (lane == 0) k = atomicAdd(P.claim + 16u + asked, 1u);
        ++asked;
        ask_at = asked < 4u ? 2 * ask_at : 0x7FFFFFFF;
        return __builtin_amdgcn_readfirstlane(k) < P.retire_most;
    };
    // kappa and Ib of a ray's (band, g) rows at a field value (sliced tables:
    // rows by LDS word, the value is the table coordinate within the
    // slice, below its last node)
    auto table_nodes = [&](float T, int kr, int ir, float& k0, float& k1, float& i0, float& i1) -> float {
        if (TAB == kTabSliced) {
            const int w = (int)T;
            lfloat* kp = (lfloat*)(uintptr_t)((uint32_t)(kr + w) << 2);
            lfloat* ip = (lfloat*)(uintptr_t)((uint32_t)(ir + w) << 2);
            k0 = kp[0];
            k1 = kp[1];
            i0 = ip[0];
            i1 = ip[1];
            return __builtin_amdgcn_fractf(T);
        }
        float pos = fmaf(T, P.inv_dT, P.mT0);
        pos = fminf(fmaxf(pos, 0.0f), (float)(nT - 1));
        int w = (int)pos;
        w = w > nT - 2 ? nT - 2 : w;
        k0 = kq[kr + w];
        k1 = kq[kr + w + 1];
        i0 = ibt[ir + w];
        i1 = ibt[ir + w + 1];
        return pos - (float)w;
    };
    auto table_at = [&](float T, int kr, int ir, float& kap, float& ibj) {
        if (SPEC == kSpecGreyT4) {
            const float t2 = T * T;
            kap = P.kappa_grey;
            ibj = t2 * t2;
            return;
        }
        float k0, k1, i0, i1;
        const float fr = table_nodes(T, kr, ir, k0, k1, i0, i1);
        kap = fmaf(fr, k1 - k0, k0);
        ibj = fmaf(fr, i1 - i0, i0);
    };
    // adaptive mesh coarsening (code/mc_gpu.cu:193-207): the lane's ray goes on
    // in the next coarser level
    auto coarser = [&]() {
        const int* F = s_lev + lev * kLevWords;
        const int* L = F + kLevWords;
        ++lev;
        maxs = L[6];
        Tl = lev_T(L);
        if (GEN) Tl += (size_t)rsnap * (uint32_t)L[14];
        // ic = (ic + r - 1) / r with r = 2 (0-based: half): every level halves
        // each axis (level g has n >> g cells)
        auto down = [&](int a, int& A, int& K, int s, float& f) {
            A = L[3 + a] + ((cell_of(F, a, A, s) >> 1) << 2) + (s > 0 ? 4 : 0);
            K = L[11 + a] + (s > 0 ? -4 : 0);
            f = lds_f(A);
        };
        down(0, A0, K0, s0, fx);
        down(1, A1, K1, s1, fy);
        down(2, A2, K2, s2, fz);
        Tc = load_T(Tl, lds_i(A0 + K0) + lds_i(A1 + K1) + lds_i(A2 + K2));
        cnt = 0;
    };

    for (;;) {
        const bool idle = !alive;
        const unsigned long long m_idle = __ballot(idle);
        const int ni = __popcll(m_idle);
        const int na = 64 - ni;
        const bool have_rays = more || cur < cend || ghead < gn || (int)cand < 0;
        // nothing left to hand out and few rays alive: the drain follows them
        // (on the last level; coarsening has few crossings before it)
        if (!have_rays && na <= kQuads && (!AMC || !__ballot(alive && lev + 1 < P.nlev))) break;
        if (have_rays && (ni >= P.refill_k || na == 0)) {
            // ---- tally the rays finished since the last refill
            if (!QUEUE && TMODE == 0) flush_wave(P, fin && rslot != aslot && aslot >= 0, aslot, aE, aA, aQ, lane);
            if (wide) ring_tally_wave(fin, rw * Dfin, rwi * G);
            if (fin) {
                rsteps = s_lev[lev * kLevWords + 15] + cnt;   // (each finer level took its maxs)
                if (QUEUE) {
                    if (!wide) ring_tally(rw * Dfin, rwi * G);
                } else
                    tally_ray<TMODE>(P, rw * Dfin, rwi * G, rslot, qcur, aslot, aE, aA, aQ);
                if (REC && qcur < P.nrec) {
                    P.rec_steps[qcur] = rsteps;
                    P.rec_end[qcur] = endt;
                    P.rec_hash[qcur] = hash;
                    P.rec_D[qcur] = Dfin;
                    P.rec_G[qcur] = G;
                }
                steps_lane += (uint32_t)rsteps;
                fin = false;
            }
            // idle lanes below this one (mbcnt: no lane mask held in registers)
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m_idle >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)m_idle, 0u));
            // the drawn ray rd of snapshot rsn becomes this lane's ray
            auto start_ray = [&](const RayStart& rd, uint32_t rsn) {
                rsnap = rsn;
                rslot = rd.six + (int)rsnap * P.tally_stride;
                if (GEN) T0 = lev_T(s_lev) + (size_t)rsnap * (uint32_t)s_lev[14];
                Tc = rd.Tc;
                band = rd.bg & 0xFFFF;
                const int fl = rd.bg >> 24;
                sx = rd.sx; sy = rd.sy; sz = rd.sz;
                ix = rd.ix; iy = rd.iy; iz = rd.iz;
                rw = rd.rw;
                rwi = rd.rwi;
                const int g = (rd.bg >> 16) & 0xFF;
                px = rd.px;
                py = rd.py;
                pz = rd.pz;
                pslot = rd.ps;
                if (AMC) {
                    lev = 0;
                    maxs = s_lev[6];
                }
                Tl = T0;
                s0 = fl & 1 ? -4 : 4;
                s1 = fl & 2 ? -4 : 4;
                s2 = fl & 4 ? -4 : 4;
                A0 = f00 + ((rd.cell & 1023) << 2) + (fl & 1 ? 0 : 4);
                A1 = f01 + (((rd.cell >> 10) & 1023) << 2) + (fl & 2 ? 0 : 4);
                A2 = f02 + (((rd.cell >> 20) & 1023) << 2) + (fl & 4 ? 0 : 4);
                K0 = k00 + (fl & 1 ? 0 : -4);
                K1 = k01 + (fl & 2 ? 0 : -4);
                K2 = k02 + (fl & 4 ? 0 : -4);
                fx = lds_f(A0);
                fy = lds_f(A1);
                fz = lds_f(A2);
                tau = 0.0f;
                tra = 1.0f;
                G = 0.0f;
                krow = kr0 + (band * P.nQ + g) * rowlen;
                ibrow = ir0 + band * rowlen;
                cnt = 0;
                hash = 2166136261u;
                alive = true;
            };
            if (QUEUE) {
                // ---- from the wave's queue of drawn rays: queue lane j holds ray
                // gbase + j of snapshot gsnap (j < gn), and the idle lane of rank r
                // takes queue lane ghead + r.  An exhausted queue is redrawn (or
                // re-read from the descriptors) for the next (up to) 64 rays of the
                // claimed super-chunk, one ray per lane, so that work runs on whole
                // waves rather than on the idle lanes of each refill.
                const uint32_t t1 = min((uint32_t)ni, gn - ghead);
                {
                    const bool s1 = idle && rank < t1;
                    const RayStart rd = pull_ray(Qr, (int)((ghead + (s1 ? rank : 0u)) & 63u));
                    if (s1 && (GEN != 1 || rd.bg >= 0)) start_ray(rd, gsnap);
                }
                ghead += t1;
                if (t1 < (uint32_t)ni) {
                    bool drawn = false;
                    if (GEN == 1 && (int)cand < 0 && retire()) {
                        more = false;
                        cand &= 0x7FFFFFFFu;
                    }
                    if (GEN == 1 && (int)cand < 0) {
                        // the next (up to) 64 listed long rays, all of the last
                        // snapshot, from this XCD's list first; no ring entries (their
                        // slots are scattered): they tally to their slots, or to an
                        // entry that holds the same slot
                        const KArgs* K = kernel_args();
                        while ((int)cand < 0) {
                            const uint32_t X = (xcd + (cand & 15u)) & 7u;
                            const uint32_t n = __builtin_amdgcn_readfirstlane(K->cand_cnt[64u * X]);
                            uint32_t c0 = 0;
                            if (lane == 0) c0 = atomicAdd(K->cand_cnt + 64u * X + 32u, 64u);
                            c0 = __builtin_amdgcn_readfirstlane(c0);
                            if (c0 >= n) {   // used up: the next list, or none left
                                cand = (cand & 15u) == 7u ? (cand & 0x7FFFFFFFu) : cand + 1u;
                                continue;
                            }
                            gn = min(64u, n - c0);
                            gsnap = (uint32_t)K->nsnap_launch - 1u;
                            if (lane == 0) atomicAdd(K->nsteps + 1, (unsigned long long)gn);   // rays listed
                            if ((uint32_t)lane < gn)
                                Qr = draw_ray(K->cand[(size_t)X * K->cand_cap + c0 + (uint32_t)lane], gsnap, true);
                            drawn = true;
                            break;
                        }
                    }
                    if (!drawn && cur >= cend && more && retire()) {
                        more = false;
                        cand &= 0x7FFFFFFFu;
                    }
                    if (!drawn && cur >= cend && more) {
                        // claim the next super-chunk, from this XCD's share first,
                        // then from the following XCDs' shares.  Claim c of XCD X is
                        // chunk X*per_x + c % per_x of snapshot c / per_x.
                        bool got = false;
                        while (xi < nparts) {
                            const uint32_t X = (xcd + xi) % nparts;
                            const uint32_t c = claim_of(X);
                            if (c >= nclaim) {
                                ++xi;
                                continue;
                            }
                            const uint32_t sn = c / per_x;
                            const uint32_t lc = X * per_x + (c - sn * per_x);
                            if (lc >= cps) continue;   // past the snapshot's last chunk
                            last_c = c;
                            csnap = sn;
                            cur = lc * S;
                            cend = cur + S < nrays ? cur + S : nrays;
                            got = true;
                            break;
                        }
                        if (!got) more = false;
                    }
                    if (drawn || cur < cend) {
                      if (!drawn) {
                        gn = min(64u, cend - cur);
                        gsnap = csnap;
                        if (GEN == 2) {
                            // the learned draws of rays cur .. cur + gn - 1: for each
                            // processing slot among them (wave-uniform) its proposal
                            // row in the wave's row buffer (evaluated unless it is the
                            // row the buffer holds), then the rays of that slot search it
                            const uint32_t q = cur + min((uint32_t)lane, gn - 1u);
                            const uint32_t slot = fdiv(q, P.fd_R);
                            const uint32_t r = q - slot * (uint32_t)P.rays_per_slot;
                            const int4 si = P.slotinfo[P.slot0 + slot];
                            const uint32_t snapshot = (uint32_t)P.snap + gsnap;
                            const u32x4 x = philox4x32_10(u32x4{r, (uint32_t)si.y, snapshot, 1u}, (uint32_t)P.seed,
                                                          (uint32_t)(P.seed >> 32));
                            const uint32_t s0 = readlane_u(slot, 0), s1 = readlane_u(slot, (int)gn - 1);
                            lr_band = 0; lr_g = 0; lr_mt = 0; lr_mp = 0; lr_ratio = 0.f;
                            // the network's arguments are read from the kernel
                            // argument segment here, not kept in registers through
                            // the traversal
                            const KArgs* K = kernel_args();
                            float* const row_buf = K->lrow_cache + (size_t)wave_id * (size_t)kLRowFloats;
                            for (uint32_t sl = s0; sl <= s1; ++sl) {
                                if (sl != row_slot || gsnap != row_snap) {
                                    learned_row(K->mlpw.W1, K->mlpw.b1, K->mlpw.W2, K->mlpw.b2, K->mlpw.W3, K->mlpw.b3,
                                                K->mlpw.nbin, K->mlpw.noutp,
                                                K->feat.T0 + (size_t)snapshot * (size_t)K->feat_stride, K->feat.n[0],
                                                K->feat.n[1], K->feat.n[2], K->feat.nbx, K->feat.nby, K->feat.centres,
                                                K->feat.coff[0], K->feat.coff[1], K->feat.coff[2], K->feat.bc_periodic,
                                                K->feat.polar, K->feat.Lpolar, K->feat.inv_Tmax, K->feat.Tw_rel,
                                                P.slotinfo[P.slot0 + sl].w, lane, row_buf);
                                    row_slot = __builtin_amdgcn_readfirstlane(sl);
                                    row_snap = __builtin_amdgcn_readfirstlane(gsnap);
                                    // the row's columns were written by every lane of the wave
                                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                                    if (K->log_rows) {
                                        const int no = K->mlpw.noutp;
                                        float* lr = K->log_rows + (size_t)(P.slot0 + sl) * (size_t)no;
                                        for (int cc = lane; cc < no; cc += 64) lr[cc] = row_buf[cc];
                                    }
                                }
                                if (slot == sl) {
                                    float qd, qb;
                                    int d, bg;
                                    mix_search2(row_buf, K->pdir, kMlpDir, row_buf + kMlpDir, K->pcdf, K->mlpw.nbin,
                                                K->mix_eps, u01_open(x.x), u01_open(x.y), &d, &qd, &bg, &qb);
                                    lr_band = bg / P.nQ;
                                    lr_g = bg - lr_band * P.nQ;
                                    lr_ratio = (qb > 0.f && qd > 0.f) ? (K->p_bg[bg] / qb) * ((1.0f / kMlpDir) / qd) : 0.f;
                                    // direction bin d = 8 cos(theta) bins x 8 phi bins: the bin in
                                    // the top 3 of the 24 uniform bits, the Philox bits below
                                    lr_mt = ((uint32_t)(d >> 3) << 21) | (x.z >> 11);
                                    lr_mp = ((uint32_t)(d & 7) << 21) | (x.w >> 11);
                                }
                            }
                            if (K->log_w0 && (uint32_t)lane < gn) {
                                uint32_t w0, w1;
                                desc_pack(lr_mt, lr_mp, lr_band, lr_g, &w0, &w1);
                                const size_t o = (size_t)gsnap * (size_t)P.nrays + (cur + (uint32_t)lane);
                                K->log_w0[o] = w0;
                                K->log_w1[o] = w1;
                                K->log_w[o] = lr_ratio;
                            }
                        }
                        if ((uint32_t)lane < gn) Qr = draw_ray(cur + (uint32_t)lane, gsnap, false);
                        cur += gn;
                        // ring entries for the batch's processing slots (consecutive:
                        // lane 0's to lane gn-1's); an entry still holding an older
                        // slot hands its sums over first (its rays still in flight
                        // then tally straight to the tally slot)
                        const int ps0 = __shfl(Qr.ps, 0), ps1 = __shfl(Qr.ps, (int)gn - 1);
                        for (int sp = ps0; sp <= ps1; ++sp) {
                            const int e = rb + (sp & (kRing - 1));
                            const int held = s_rt[e];
                            if (held == sp) continue;
                            const unsigned long long mine = __ballot((uint32_t)lane < gn && Qr.ps == sp);
                            const int tgt = __shfl(Qr.six, __ffsll((long long)mine) - 1) + (int)gsnap * P.tally_stride;
                            if (lane == 0) {
                                if (held >= 0) ring_flush(e);
                                s_rt[e] = sp;
                                s_rg[e] = tgt;
                                s_rv[3 * e] = s_rv[3 * e + 1] = s_rv[3 * e + 2] = 0.0;
                            }
                        }
                      }
                        const bool s2 = idle && rank >= t1 && rank - t1 < gn;
                        const RayStart rd = pull_ray(Qr, (int)(s2 ? rank - t1 : 0u));
                        if (s2 && (GEN != 1 || rd.bg >= 0)) start_ray(rd, gsnap);
                        ghead = min((uint32_t)ni - t1, gn);
                    }
                }
            } else {
                // ---- hand out consecutive rays to the idle lanes, in lane order
                const uint32_t avail = cend - cur;
                uint32_t q = 0xFFFFFFFFu, qs = csnap;
                if (idle && rank < avail) q = cur + rank;
                if (avail < (uint32_t)ni && more && retire()) more = false;
                if (avail < (uint32_t)ni && more) {
                    // the current super-chunk runs out: claim the next one (as above)
                    bool got = false;
                    uint32_t nstart = 0, nend = 0, nsn = 0;
                    while (xi < nparts) {
                        const uint32_t X = (xcd + xi) % nparts;
                        const uint32_t c = claim_of(X);
                        if (c >= nclaim) {
                            ++xi;
                            continue;
                        }
                        const uint32_t sn = c / per_x;
                        const uint32_t lc = X * per_x + (c - sn * per_x);
                        if (lc >= cps) continue;   // past the snapshot's last chunk
                        last_c = c;
                        nsn = sn;
                        nstart = lc * S;
                        nend = nstart + S < nrays ? nstart + S : nrays;
                        got = true;
                        break;
                    }
                    if (got) {
                        if (idle && rank >= avail && nstart + (rank - avail) < nend) {
                            q = nstart + (rank - avail);
                            qs = nsn;
                        }
                        const uint32_t used = (uint32_t)ni - avail;
                        cur = nstart + used < nend ? nstart + used : nend;
                        cend = nend;
                        csnap = nsn;
                    } else {
                        more = false;
                        cur = cend;
                    }
                } else {
                    cur += avail < (uint32_t)ni ? avail : (uint32_t)ni;
                }
                // ---- start the handed-out rays
                if (q != 0xFFFFFFFFu) {
                    qcur = q;
                    start_ray(draw_ray(q, qs, false), qs);
                }
            }
        }
        if (!alive) continue;

        // ------------------------------------------------ kAhead crossings
        constexpr int kAhead = AMC ? kAheadLev : kAheadFine;
        float dsv[kAhead], Tv[kAhead];
        int lin[kAhead];
        const int lim = AMC ? min(kAhead, maxs - cnt) : kAhead;
        int wall = -1, wall_u = kAhead;         // the crossing that hits a wall
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            dsv[u] = Tv[u] = 0.0f;
            lin[u] = 0;
            if (AMC && u >= lim) continue;
            if (REC) {
                const int* L = s_lev + lev * kLevWords;
                lin[u] = cell_of(L, 0, A0, s0) + L[0] * (cell_of(L, 1, A1, s1) + L[1] * cell_of(L, 2, A2, s2));
            }
            const float d0 = (fx - px) * ix;
            const float d1 = (fy - py) * iy;
            const float d2 = (fz - pz) * iz;
            const float ds = min3(d0, d1, d2);
            dsv[u] = ds;
            const bool e0 = ds == d0, e1 = ds == d1, m2 = ds == d2;
            px = e0 ? fx : fmaf(ds, sx, px);
            py = e1 ? fy : fmaf(ds, sy, py);
            pz = m2 ? fz : fmaf(ds, sz, pz);
            // of several axes at the same distance the last one moves
            const bool m1 = e1 && !m2, m0 = e0 && !e1 && !m2;
            A0 += m0 ? s0 : 0;
            A1 += m1 ? s1 : 0;
            A2 += m2 ? s2 : 0;
            float fnew = lds_f(m2 ? A2 : (m1 ? A1 : A0));
            // (read with the face: one LDS latency before the field load; a ray that
            // left the domain reads its neighbours' words here and its own below)
            int o0 = lds_i(A0 + K0), o1 = lds_i(A1 + K1), o2 = lds_i(A2 + K2);
            asm volatile("" : "+v"(fnew), "+v"(o0), "+v"(o1), "+v"(o2));   // (here, not sunk past the branch)
            // past the domain's last face: a periodic wrap, or a wall hit that keeps
            // the old cell (the ray ends there).  Rare per lane, so a branch.
            if (fnew > kFaceEnd * 0.5f) {
                const int ax = m2 ? 2 : (m1 ? 1 : 0);
                const int sa = m2 ? s2 : (m1 ? s1 : s0);
                const int side = sa > 0 ? 1 : 0;
                const int bcbit = ax * 2 + side;
                const int* L = s_lev + lev * kLevWords + ax;
                const int fo = L[3], last = fo + (L[0] << 2);     // face 0, face n
                int An = (m2 ? A2 : (m1 ? A1 : A0)) - sa;
                if ((P.bc_periodic >> bcbit) & 1) {
                    const float pw = lds_f(side ? fo : last);
                    An = side ? fo + 4 : last - 4;
                    px = m0 ? pw : px;
                    py = m1 ? pw : py;
                    pz = m2 ? pw : pz;
                } else if (wall < 0) {
                    wall = bcbit;
                    wall_u = u;
                }
                A0 = m0 ? An : A0;
                A1 = m1 ? An : A1;
                A2 = m2 ? An : A2;
                fnew = lds_f(An);
                o0 = lds_i(A0 + K0);
                o1 = lds_i(A1 + K1);
                o2 = lds_i(A2 + K2);
            }
            fx = m0 ? fnew : fx;
            fy = m1 ? fnew : fy;
            fz = m2 ? fnew : fz;
            Tv[u] = load_T(Tl, o0 + o1 + o2);
        }
        // transport, branch-free on the common path: past the cut-off the
        // remaining energy is deposited here (tra), else the segment absorbs
        // tra - tra1; a wall absorbs what is left; the step cap ends the ray
        // (or moves it to the next coarser level)
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (!alive || (AMC && u >= lim)) continue;
            float kap, ibj;
            table_at(Tc, krow, ibrow, kap, ibj);
            if (REC) hash = (hash ^ (((uint32_t)lev << 28) ^ (uint32_t)lin[u])) * 16777619u;
            ++cnt;
            Tc = Tv[u];
            tau = fmaf(kap, dsv[u], tau);
            const bool cut = tau >= P.tau_cut, hit = u == wall_u;
            const float tra1 = __expf(-tau);
            G = fmaf(cut ? tra : tra - tra1, ibj, G);
            tra = tra1;   // (not used after a cut-off)
            if (cut || hit || cnt >= maxs) {
                if (cut || hit) {
                    if (!cut) G = fmaf(tra, s_ibw[wall * P.nB + band], G);
                    alive = false; fin = true; endt = cut ? 0 : 1; Dfin = 1.0f;
                } else if (!AMC || lev + 1 >= P.nlev) {
                    alive = false; fin = true; endt = 2; Dfin = 1.0f - tra;
                }
            }
        }
        if (AMC && alive && cnt >= maxs) coarser();
    }
    // ---- drain: nothing is left to hand out and at most 16 of the wave's rays
    // run on, on the last level.  Such a ray is a serial chain (along the walls
    // in a thin bin up to the step cap, 1e5 crossings): one crossing per
    // iteration of the loop above takes 350 ns, 840 cycles, of which 380 issue
    // its 95 instructions and the rest waits for LDS and the field; a
    // 64x96x64 solve of 2e8 rays spent 36 of its 46 ms here.  So four lanes
    // follow one ray.  The cells a ray crosses do not depend on the field:
    // lane a of the quad holds axis a (lane 3 none) and the quad moves kDrain
    // crossings ahead, the nearest face by quad permutes, the two faces behind
    // the exit face read ahead.  Then the batch's field loads and table
    // lookups run in parallel, crossing 4 k + j on lane j, and tau and G
    // follow in crossing order with the main loop's arithmetic (a crossing
    // past the ray's end has length 0 and adds 0): 122 ns per crossing with
    // a branch per crossing for walls, wraps and ties, 105 ns without (below):
    // a launch bound by one ray of 16000 crossings 2.23 -> 2.04 ms.  Batches of
    // 8, 16, 24 and 32 crossings: 2.34, 2.03, 2.18 and 2.22 ms there.  The
    // first solve 46 -> 22 ms (18 with retiring waves, above).
    if (__ballot(alive)) {
        __builtin_amdgcn_s_setprio(3);   // ahead of the waves that still trace the bulk
        const unsigned long long am = __ballot(alive);
        const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(am >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)am, 0u));
        // the lane of the ray that this quad follows: its rank-th alive lane
        // (each alive lane sends its number to lane 4 rank, the others to 63)
        int src = quad_i<0>(__builtin_amdgcn_ds_permute(alive ? 16 * rank : 4 * 63, lane));
        const int a = lane & 3;
        const bool ax3 = a == 3;
        bool run = (lane >> 2) < __popcll(am);
        src = run ? src : 0;
        auto axis_f = [&](float x, float y, float z, float w) -> float {
            const float vx = __shfl(x, src), vy = __shfl(y, src), vz = __shfl(z, src);
            return a == 0 ? vx : (a == 1 ? vy : (a == 2 ? vz : w));
        };
        // (lane 3 is never the nearest face: distance 3e38)
        float qp = axis_f(px, py, pz, 0.0f), qs = axis_f(sx, sy, sz, 0.0f), qi = axis_f(ix, iy, iz, 1.0f);
        float qf = axis_f(fx, fy, fz, 3.0e38f);
        const bool neg = axis_f(sx, sy, sz, 1.0f) < 0.0f;
        const int* L = s_lev + (P.nlev - 1) * kLevWords; // the last level
        int qc;                                          // 0-based cell
        {
            const int vx = __shfl(A0, src), vy = __shfl(A1, src), vz = __shfl(A2, src);
            // (a quad without a ray stays frozen in cell 0: lane 0's last ray may
            // have ended on a finer level, whose cells this level does not have)
            qc = !run || ax3 ? 0 : cell_of(L, a, a == 0 ? vx : (a == 1 ? vy : vz), neg ? -4 : 4);
        }
        const int st = neg ? -1 : 1;
        float qtau = __shfl(tau, src), qtra = __shfl(tra, src), qG = __shfl(G, src);
        const int qkrow = __shfl(krow, src), qibrow = __shfl(ibrow, src), qband = __shfl(band, src);
        int qcnt = __shfl(cnt, src), qend = 0;
        float qD = 1.0f;
        uint32_t qhash = REC ? (uint32_t)__shfl((int)hash, src) : 0u;
        const int bcbit = 2 * a + (neg ? 0 : 1);         // the boundary this axis runs into
        const bool per = (P.bc_periodic >> bcbit) & 1;
        // cells along this axis, LDS bytes of the face behind the exit face of
        // cell 0 and of its brick offset
        const int qn = ax3 ? 0x7FFFFFFF : L[a], qmaxs = L[6];
        const int gb = L[3 + (ax3 ? 0 : a)] + (neg ? -4 : 8), ob = L[3 + (ax3 ? 0 : a)] + L[11 + (ax3 ? 0 : a)];
        const int qstride = a == 0 ? 1 : (a == 1 ? L[0] : (a == 2 ? L[0] * L[1] : 0));
        gfloat* qT = lev_T(L);
        if (GEN) qT += (size_t)(uint32_t)__shfl((int)rsnap, src) * (uint32_t)L[14];
        // face i behind (+) or before (-) the exit face of cell c: word c + i st of
        // the face table from gb - st (a word past the axis's faces is one of its
        // LDS neighbours and is not used)
        auto face_w = [&](int byte, int i) -> float { return lds_f(byte + (i << 2)); };
        // the walk's per-lane constants (lane 3: one cell, never left): the
        // cell behind the domain's last (the other end's, or out of range at a
        // wall) and the coordinate there
        const uint32_t wn = ax3 ? 1u : (uint32_t)qn;
        const int wrapc = ax3 ? 0 : (per ? (neg ? qn - 1 : 0) : (neg ? -1 : qn));
        const float wrapp = per && !ax3 ? face_w(gb - 4 * st - (neg ? 0 : 4), neg ? qn : 0) : 0.0f;
        const int xb = gb - 4 * st;                      // exit face of cell 0
        while (__ballot(run)) {
            int lim = run ? min(kDrain, qmaxs - qcnt) : 0;
            int wall = -1;
            // (a quad without a running ray moves within the domain, or not at all,
            // and its crossings have length 0)
            qc = run ? qc : 0;
            qs = run ? qs : 0.0f;
            qi = run ? qi : 0.0f;
            float dsv[kDrain], Tv[kDrain / 4];
            int lin[kDrain / 4];
            // The walk, without a branch and with nothing through scalar registers: a
            // lane moves when its face is the nearest, wraps and walls follow from
            // its cell (past a wall the face is at 3e38 and the cell stays out of
            // range: nout counts the crossings since).  Axes that tie show in the
            // number of moves; the batch is then walked again, the last of them
            // moving first.
            const float qp0 = qp, qf0 = qf;
            const int qc0 = qc;
            int nout, nm;
            for (bool careful = false;; careful = true) {
                nout = nm = 0;
                auto behind = [&](int c, bool& out) -> int {
                    out = (uint32_t)(c + st) >= wn;
                    return out ? wrapc : c + st;
                };
                bool o1, o2;
                int cn = behind(qc, o1);
                float qa = o1 ? wrapp : qf;              // the coordinate behind the exit face
                float g = face_w(xb, cn);
                float h = face_w(xb, behind(cn, o2));
#pragma unroll
                for (int k = 0; k < kDrain / 4; ++k) {
                    int ov[4];
                    lin[k] = 0;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int u = 4 * k + j;
                        ov[j] = lds_i(ob + (int)(min((uint32_t)qc, wn - 1u) << 2));
                        const float d = (qf - qp) * qi;
                        const float ds = quad_min(d);
                        dsv[u] = ds;
                        bool mv = d == ds, tie = false;
                        if (__builtin_expect(careful, 0)) {
                            const int e = mv ? 1 : 0;
                            tie = (e & (quad_i<0xF9>(e) | quad_i<0xFE>(e))) != 0;   // (lanes a + 1 and a + 2)
                            mv = mv && !tie;
                        }
                        if (REC) {
                            const int l = quad_sum(qc * qstride);
                            lin[k] = a == j ? l : lin[k];
                        }
                        const float pn = tie ? qf : fmaf(ds, qs, qp);
                        qp = mv ? qa : pn;
                        nm += mv ? 1 : 0;
                        qf = mv ? g : qf;
                        g = mv ? h : g;
                        qc = mv ? cn : qc;
                        nout += (uint32_t)qc >= wn ? 1 : 0;
                        cn = behind(qc, o1);
                        qa = o1 ? wrapp : qf;
                        h = face_w(xb, behind(cn, o2));
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) ov[j] = ax3 ? 0 : ov[j];   // (here, not on the chain: the reads have come)
                    Tv[k] = load_T(qT, quad_spread(ov, a));
                }
                if (careful || !__ballot(run && quad_sum(nm) != kDrain)) break;
                qp = qp0;
                qf = qf0;
                qc = qc0;
            }
            if (__ballot(nout > 0 && run)) {
                // the first wall of the batch, if it comes before the step cap
                const int uh = kDrain - nout, um = quad_min_i(uh);
                const int w = quad_max(nout > 0 && uh == um ? bcbit : -1);
                wall = um < lim ? w : -1;
                lim = min(lim, um + 1);
            }
            if (__ballot(run && lim < kDrain)) {             // the step cap inside the batch
#pragma unroll
                for (int u = 0; u < kDrain; ++u) dsv[u] = u < lim ? dsv[u] : 0.0f;
            }
            // the lookups
            float kap[kDrain / 4], ibv[kDrain / 4], tk[kDrain / 4], dg[kDrain / 4];
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) table_at(Tv[k], qkrow, qibrow, kap[k], ibv[k]);
            // optical depth in crossing order (every lane of the quad), kept by
            // the crossing's lane
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                float t[4];
                quad_fma_t(qtau, kap[k], dsv + 4 * k, t);
                tk[k] = a == 0 ? t[0] : (a == 1 ? t[1] : (a == 2 ? t[2] : t[3]));
            }
            // transmissivities; the first crossing past the cut-off
            int first = kDrain;
            float before = qtra;   // transmissivity before this group of four
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                const bool cut = tk[k] >= P.tau_cut;
                const float t1 = __expf(-tk[k]);
                const float t0 = quad_f<kQuadPrev>(t1);      // (every lane of the quad takes part)
                const float tp = a == 0 ? before : t0;
                dg[k] = cut ? tp : tp - t1;
                first = min(first, cut ? 4 * k + a : kDrain);
                before = quad_f<0xFF>(t1);
            }
            bool cutq = false;
            int taken = lim;
            if (__ballot(first < lim)) {
                first = quad_min_i(first);
                cutq = first < lim;
                taken = cutq ? first + 1 : lim;
#pragma unroll
                for (int k = 0; k < kDrain / 4; ++k) dg[k] = 4 * k + a < taken ? dg[k] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                quad_fma(qG, dg[k], quad_f<0x00>(ibv[k]), quad_f<0x55>(ibv[k]), quad_f<0xAA>(ibv[k]), quad_f<0xFF>(ibv[k]));
            }
            if (REC) {
                const uint32_t lb = (uint32_t)(P.nlev - 1) << 28;
#pragma unroll
                for (int k = 0; k < kDrain / 4; ++k) {
                    const uint32_t l0 = (uint32_t)quad_i<0x00>(lin[k]), l1 = (uint32_t)quad_i<0x55>(lin[k]);
                    const uint32_t l2 = (uint32_t)quad_i<0xAA>(lin[k]), l3 = (uint32_t)quad_i<0xFF>(lin[k]);
                    if (4 * k < taken) qhash = (qhash ^ (lb ^ l0)) * 16777619u;
                    if (4 * k + 1 < taken) qhash = (qhash ^ (lb ^ l1)) * 16777619u;
                    if (4 * k + 2 < taken) qhash = (qhash ^ (lb ^ l2)) * 16777619u;
                    if (4 * k + 3 < taken) qhash = (qhash ^ (lb ^ l3)) * 16777619u;
                }
            }
            qtra = before;   // (not used after a cut-off)
            qcnt += taken;
            const bool hitw = run && !cutq && wall >= 0;
            if (hitw) qG = fmaf(qtra, s_ibw[wall * P.nB + qband], qG);
            if (run && (cutq || hitw)) {
                run = false;
                qend = cutq ? 0 : 1;
                qtau = 0.0f;   // (the quad idles below the cut-off: it adds 0)
                qtra = 1.0f;
            } else if (run && qcnt >= qmaxs) {
                run = false;
                qend = 2;
                qD = 1.0f - qtra;
            }
        }
        // back to the lanes that held the rays
        const int from = alive ? 4 * rank : lane;
        const float rG = __shfl(qG, from), rD = __shfl(qD, from);
        const int rcn = __shfl(qcnt, from), ren = __shfl(qend, from);
        const uint32_t rh = REC ? (uint32_t)__shfl((int)qhash, from) : 0u;
        if (alive) {
            G = rG;
            Dfin = rD;
            cnt = rcn;
            endt = ren;
            if (REC) hash = rh;
            alive = false;
            fin = true;
        }
        __builtin_amdgcn_s_setprio(0);
    }
    // a ray that ended after the last refill (nothing was left to hand out)
    if (!QUEUE && TMODE == 0) flush_wave(P, fin && rslot != aslot && aslot >= 0, aslot, aE, aA, aQ, lane);
    if (fin) {
        rsteps = s_lev[lev * kLevWords + 15] + cnt;
        if (QUEUE)
            ring_tally(rw * Dfin, rwi * G);
        else
            tally_ray<TMODE>(P, rw * Dfin, rwi * G, rslot, qcur, aslot, aE, aA, aQ);
        if (REC && qcur < P.nrec) {
            P.rec_steps[qcur] = rsteps;
            P.rec_end[qcur] = endt;
            P.rec_hash[qcur] = hash;
            P.rec_D[qcur] = Dfin;
            P.rec_G[qcur] = G;
        }
        steps_lane += (uint32_t)rsteps;
    }
    if (!QUEUE && TMODE == 0) flush_wave(P, aslot >= 0, aslot, aE, aA, aQ, lane);
    // the ring's remaining sums
    if (QUEUE && lane < kRing && s_rt[rb + lane] >= 0) ring_flush(rb + lane);
    // one step-count atomic per wave
    unsigned long long st = steps_lane;
    for (int off = 32; off > 0; off >>= 1) st += __shfl_xor(st, off);
    if (lane == 0) atomicAdd(P.nsteps, st);
}

// ------------------------------------------------------------ trace_f64 ----
// FP64 traversal (precision 1, plain estimator): every ray in double, as the
// FP64 oracle computes it.  Direction from the descriptor's 24-bit uniforms,
// table lookups interpolated in FP64 from the FP32 tables, FP64 optical depth,
// transmissivity and gathered emission, bundle weights recomputed in FP64:
// w = Ibmax (k_i Ib_i) / (k_max Ib_max), E = w D, A = w G / Ib_i; each ray's
// (E, A) goes to pray64 for reduce_rays.
__device__ __forceinline__ void lookup_f64(const TraceArgs& P, double Tj, int bg, int band, double* kap, double* ib)
{
    double pos = Tj * (double)P.inv_dT + (double)P.mT0;
    pos = pos < 0.0 ? 0.0 : pos;
    pos = pos > (double)(P.nT - 1) ? (double)(P.nT - 1) : pos;
    int t0 = (int)pos;
    t0 = t0 > P.nT - 2 ? P.nT - 2 : t0;
    const double fr = pos - (double)t0;
    const float* kr = P.kq + (size_t)bg * P.nT;
    const float* ir = P.Ib + (size_t)band * P.nT;
    *kap = (double)kr[t0] + fr * ((double)kr[t0 + 1] - (double)kr[t0]);
    *ib = (double)ir[t0] + fr * ((double)ir[t0 + 1] - (double)ir[t0]);
}

__device__ __forceinline__ double min_f64(double x, double y)   // (no NaN)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
__device__ __forceinline__ double quad_min_d(double v)
{
    v = min_f64(v, quad_d<kQuadXor1>(v));
    return min_f64(v, quad_d<kQuadXor2>(v));
}

// Work (LONG): the rays are cut into a share per XCD; a wave takes `super` rays
// of its XCD's share by its place, then claims as many at a time from a counter
// per share, the others' when its own is used up, and starts new rays when 16
// lanes are idle.  (One counter for all, the first chunks claimed too: its
// atomics, 11 ns each, were a quarter of a launch of 4e5 short rays: 4e5 rays of
// 3.3 crossings 0.275 -> 0.227 ms, 8e5 of 3.6 on three levels 0.545 -> 0.465.)
// The drain below is the FP32 traversal's: when nothing is
// left to hand out and at most 16 of a wave's rays run on, all on the last
// level, four lanes follow a ray, kDrain crossings ahead, with the loop's
// arithmetic and order (a crossing past the ray's end has length 0).
//
// Such a launch waits for its longest ray: one crossing after another takes
// about 700 ns here (faces, field, table and exponential one behind the other).
// 1024 cells x 8192 rays of a 64x96x64 channel, 9.1e7 crossings, longest ray
// 16000, on three temperature fields: 12.2, 8.5 and 8.8 ms with a thread per ray,
// 3.9, 2.7 and 2.7 ms with the drain (the bulk about 1 ms of it).
//
// Grey rays of few hundred crossings at most (!LONG, the host's rule) have no
// long chain among them: a thread per ray, without the drain's registers (four
// waves per SIMD instead of three).
template <int SPEC, bool REC, bool LONG>
__global__ __launch_bounds__(256, LONG ? 1 : 4) void trace_f64(TraceArgs P, double2* pray64)
{
    extern __shared__ float lds[];
    int* s_lev = (int*)lds;
    float* s_face = lds + 6 * kLevWords;
    int* s_off = (int*)(s_face + P.nfaces);
    float* s_cent = (float*)(s_off + P.noffs);
    float* s_ibw = s_cent + P.ncent;
    for (int i = threadIdx.x; i < P.nlev; i += blockDim.x) {
        int* L = s_lev + i * kLevWords;
        L[0] = P.lev[i].n[0]; L[1] = P.lev[i].n[1]; L[2] = P.lev[i].n[2];
        L[3] = P.lev[i].foff[0]; L[4] = P.lev[i].foff[1]; L[5] = P.lev[i].foff[2];
        L[6] = P.lev[i].maxs;
        const unsigned long long t = (unsigned long long)(P.T[i] + (size_t)P.snap * P.lev[i].tstride);
        L[7] = (int)(uint32_t)t; L[8] = (int)(uint32_t)(t >> 32);
        L[11] = P.lev[i].ooff[0]; L[12] = P.lev[i].ooff[1]; L[13] = P.lev[i].ooff[2];
    }
    for (int i = threadIdx.x; i < P.nfaces; i += blockDim.x) s_face[i] = P.faces[i];
    for (int i = threadIdx.x; i < P.noffs; i += blockDim.x) s_off[i] = P.offs[i];
    for (int i = threadIdx.x; i < P.ncent; i += blockDim.x) s_cent[i] = P.centres[i];
    for (int i = threadIdx.x; i < 6 * P.nB; i += blockDim.x) s_ibw[i] = P.Ibw[i];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const double Tm = (double)P.Tmax, tau_cut = (double)P.tau_cut;
    unsigned long long steps_t = 0;
    // the lane's ray
    bool alive = false;
    uint32_t q = 0;
    int f[3], c[3], band = 0, bg = 0, lev = 0, cnt = 0, steps = 0;
    double s[3], inv[3], p[3], w = 0.0, ii = 1.0, tau = 0.0, tra = 1.0, G = 0.0;
    uint32_t hash = 0;
    // of its level
    int n[3], fo[3], oo[3], maxs = 0;
    gfloat* T = nullptr;
    for (int a = 0; a < 3; ++a) {
        f[a] = 0; c[a] = 1; n[a] = fo[a] = oo[a] = 0;
        s[a] = inv[a] = 1.0; p[a] = 0.0;
    }
    auto set_level = [&]() {
        const int* L = s_lev + lev * kLevWords;
        for (int a = 0; a < 3; ++a) {
            n[a] = L[a];
            fo[a] = L[3 + a];
            oo[a] = L[11 + a];
        }
        maxs = L[6];
        T = lev_T(L);
        cnt = 0;
    };
    auto finish = [&](double D, int endt) {
        pray64[q] = make_double2(w * D, w * G / ii);
        steps_t += (unsigned long long)steps;
        if (REC && q < P.nrec) {
            P.rec_steps[q] = steps;
            P.rec_end[q] = endt;
            P.rec_hash[q] = hash;
            P.rec_D[q] = (float)D;
            P.rec_G[q] = (float)G;
        }
        alive = false;
    };
    // the step cap: the next coarser level, or the end on the last
    auto capped = [&]() {
        while (alive && cnt >= maxs) {
            if (lev + 1 < P.nlev) {
                const int m[3] = {n[0], n[1], n[2]};
                ++lev;
                set_level();
                for (int a = 0; a < 3; ++a) {
                    const int r = m[a] / n[a];
                    c[a] = (c[a] + r - 1) / r;
                }
            } else {
                finish(1.0 - tra, 2);
            }
        }
    };
    auto start = [&]() {
        const uint32_t a0 = P.w0[q], a1 = P.w1[q];
        const int4 si = P.slotinfo[P.slot0 + fdiv(q, P.fd_R)];
        const int g = desc_g(a1);
        band = desc_band(a0, a1);
        bg = band * P.nQ + g;
        const double ut = ((double)(a0 & 0xFFFFFFu) + (double)P.u_off) * 5.9604644775390625e-08;
        const double up = ((double)(a1 & 0xFFFFFFu) + (double)P.u_off) * 5.9604644775390625e-08;
        {
            const int a = P.polar;
            const double cth = 1.0 - 2.0 * ut, st = 2.0 * sqrt(ut * (1.0 - ut));
            const double ph = 6.283185307179586476925 * up;
            const double c1 = st * cos(ph), c2 = st * sin(ph);
            s[0] = a == 0 ? cth : (a == 1 ? c2 : c1);
            s[1] = a == 0 ? c1 : (a == 1 ? cth : c2);
            s[2] = a == 0 ? c2 : (a == 1 ? c1 : cth);
        }
        for (int a = 0; a < 3; ++a) {
            if (s[a] == 0.0) s[a] = 1e-10;
            f[a] = s[a] < 0.0;
            inv[a] = 1.0 / s[a];
        }
        c[0] = (si.w & 1023) + 1;
        c[1] = ((si.w >> 10) & 1023) + 1;
        c[2] = ((si.w >> 20) & 1023) + 1;
        for (int a = 0; a < 3; ++a) p[a] = (double)s_cent[P.coff[a] + c[a]];
        const double Ti = (double)P.T[0][(size_t)P.snap * P.lev[0].tstride + si.z];
        double ki, kmx, imx;
        if (SPEC == kSpecGreyT4) {
            ki = kmx = (double)P.kappa_grey;
            ii = Ti * Ti * Ti * Ti;
            imx = Tm * Tm * Tm * Tm;
        } else {
            lookup_f64(P, Ti, bg, band, &ki, &ii);
            lookup_f64(P, Tm, bg, band, &kmx, &imx);
        }
        w = P.Ibmax_d * (ki * ii) / (kmx * imx);
        tau = 0.0;
        tra = 1.0;
        G = 0.0;
        steps = 0;
        hash = 2166136261u;
        lev = 0;
        alive = true;
        set_level();
        capped();
    };
    auto cross = [&]() {
        double fx[3], d[3];
        for (int a = 0; a < 3; ++a) {
            fx[a] = (double)s_face[fo[a] + c[a] - f[a]];
            d[a] = (fx[a] - p[a]) * inv[a];
        }
        double ds = d[0];
        ds = ds > d[1] ? d[1] : ds;
        ds = ds > d[2] ? d[2] : ds;
        for (int a = 0; a < 3; ++a) p[a] = (ds == d[a]) ? fx[a] : p[a] + ds * s[a];
        if (REC) {
            const int lin = (c[0] - 1) + n[0] * ((c[1] - 1) + n[1] * (c[2] - 1));
            hash = (hash ^ (((uint32_t)lev << 28) ^ (uint32_t)lin)) * 16777619u;
        }
        const double Tj = (double)load_T(T, s_off[oo[0] + c[0] - 1] + s_off[oo[1] + c[1] - 1] + s_off[oo[2] + c[2] - 1]);
        double kap, ibj;
        if (SPEC == kSpecGreyT4) {
            kap = (double)P.kappa_grey;
            ibj = Tj * Tj * Tj * Tj;
        } else {
            lookup_f64(P, Tj, bg, band, &kap, &ibj);
        }
        ++steps;
        ++cnt;
        const double tau1 = tau + kap * ds;
        if (tau1 >= tau_cut) {
            G += tra * ibj;
            finish(1.0, 0);
            return;
        }
        const double tra1 = exp(-tau1);
        G += (tra - tra1) * ibj;
        tau = tau1;
        tra = tra1;
        const int ax = (d[0] < d[1]) ? ((d[0] < d[2]) ? 0 : 2) : ((d[1] < d[2]) ? 1 : 2);
        for (int a = 0; a < 3; ++a) {
            if (ax != a) continue;
            c[a] += f[a] ? -1 : 1;
            if (c[a] == 0 || c[a] == n[a] + 1) {
                const int side = c[a] != 0;
                if ((P.bc_periodic >> (a * 2 + side)) & 1) {
                    c[a] = side ? 1 : n[a];
                    p[a] = (double)s_face[fo[a] + (side ? 0 : n[a])];
                } else {
                    G += tra * (double)s_ibw[(a * 2 + side) * P.nB + band];
                    finish(1.0, 1);
                }
            }
        }
        capped();
    };
    auto count_steps = [&]() {
        for (int off = 32; off > 0; off >>= 1) steps_t += __shfl_xor(steps_t, off);
        if (lane == 0) atomicAdd(P.nsteps, steps_t);
    };
    if (!LONG) {
        for (long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x; r < P.nrays; r += (long long)gridDim.x * blockDim.x) {
            q = (uint32_t)r;
            start();
            while (alive) cross();
        }
        count_steps();
        return;
    }
    // the wave's rays cb..ce: at first a chunk by its place among the waves of
    // its XCD's share, then claimed ones
    uint32_t cb = 0, ce = 0;
    auto waves = [&](uint32_t X) -> uint32_t { return ((gridDim.x + 7u - X) >> 3) * 4u; };
    // chunk c (of S rays) of share X (p rays): its waves' places come first, then
    // its counter's claims
    auto take_chunk = [&](uint32_t X, uint32_t c, uint32_t S, uint32_t nrays, uint32_t p) -> bool {
        const uint32_t n = X * p < nrays ? min(p, nrays - X * p) : 0u;
        if (c * S >= n) return false;
        cb = readlane_u(X * p + c * S, 0);
        ce = readlane_u(cb + min(S, n - c * S), 0);
        return true;
    };
    auto share = [](uint32_t nrays) -> uint32_t { return ((nrays + 7u) / 8u + 63u) / 64u * 64u; };
    uint32_t home = (blockIdx.x & 7u) | 8u;  // its XCD; bit 3 while that share may have rays left
    // one try: false when no share has rays left (cb == ce: another wave was first);
    // readlane: the compiler then keeps the hand-out in scalar registers
    auto claim = [&]() -> bool {
        const KArgs* K = kernel_args();      // (read here, not held through the traversal)
        const uint32_t nrays = (uint32_t)__builtin_amdgcn_readfirstlane((int)K->nrays);
        const uint32_t S = (uint32_t)__builtin_amdgcn_readfirstlane(K->super), p = share(nrays);
        uint32_t X = home & 7u;
        if (!(home & 8u)) {
            bool has = false;                // lane x: share x has rays left
            if (lane < 8 && lane * p < nrays)
                has = S * (waves(lane) + __hip_atomic_load(K->claim + 32 * lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) <
                      min(p, nrays - lane * p);
            const uint32_t left = readlane_u((uint32_t)__ballot(has), 0);
            if (!left) return false;
            X = (X + (uint32_t)__builtin_ctz((left | (left << 8)) >> X)) & 7u;
        }
        uint32_t c = 0;
        if (lane == 0) c = atomicAdd(K->claim + 32u * X, 1u);
        if (!take_chunk(X, waves(X) + (uint32_t)__builtin_amdgcn_readfirstlane((int)c), S, nrays, p)) home = readlane_u(home & 7u, 0);
        return true;
    };
    take_chunk(home & 7u, (blockIdx.x >> 3) * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), (uint32_t)P.super,
               (uint32_t)P.nrays, share((uint32_t)P.nrays));
    bool more = true;
    for (;;) {
        unsigned long long idle = __ballot(!alive);
        if (more && __popcll(idle) >= 16) {
            while (idle) {
                if (cb >= ce && !claim()) {
                    more = false;
                    break;
                }
                const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
                const uint32_t take = min((uint32_t)__popcll(idle), ce - cb);
                if (!alive && (uint32_t)rank < take) {
                    q = cb + (uint32_t)rank;
                    start();
                }
                cb += take;
                idle = __ballot(!alive);
            }
        }
        const unsigned long long am = __ballot(alive);
        if (!am) break;   // (nothing is left to hand out either)
        if (!more && __popcll(am) <= kQuads && !__ballot(alive && lev + 1 < P.nlev)) break;
        if (alive) cross();
    }
    // ---- drain: lane a of a quad holds axis a of its ray (lane 3 none)
    if (__ballot(alive)) {
        __builtin_amdgcn_s_setprio(3);
        const unsigned long long am = __ballot(alive);
        const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(am >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)am, 0u));
        // the lane of the ray that this quad follows: its rank-th alive lane
        // (each alive lane sends its number to lane 4 rank, the others to 63)
        int src = quad_i<0>(__builtin_amdgcn_ds_permute(alive ? 16 * rank : 4 * 63, lane));
        const int a = lane & 3;
        const bool ax3 = a == 3;
        bool run = (lane >> 2) < __popcll(am);
        src = run ? src : 0;
        auto axis_d = [&](const double* v, double w3) -> double {
            const double vx = __shfl(v[0], src), vy = __shfl(v[1], src), vz = __shfl(v[2], src);
            return a == 0 ? vx : (a == 1 ? vy : (a == 2 ? vz : w3));
        };
        const int* L = s_lev + (P.nlev - 1) * kLevWords;   // the last level
        double qp = axis_d(p, 0.0), qs = axis_d(s, 0.0), qi = axis_d(inv, 1.0);
        int qc;                                            // 0-based cell (0 where the quad has no ray)
        bool neg;
        {
            const int c0 = __shfl(c[0], src), c1 = __shfl(c[1], src), c2 = __shfl(c[2], src);
            const int f0 = __shfl(f[0], src), f1 = __shfl(f[1], src), f2 = __shfl(f[2], src);
            qc = !run || ax3 ? 0 : (a == 0 ? c0 : (a == 1 ? c1 : c2)) - 1;
            neg = a == 0 ? f0 != 0 : (a == 1 ? f1 != 0 : (a == 2 ? f2 != 0 : false));
        }
        const int st = neg ? -1 : 1;
        double qtau = __shfl(tau, src), qtra = __shfl(tra, src), qG = __shfl(G, src);
        const int qbg = __shfl(bg, src), qband = __shfl(band, src);
        int qcnt = __shfl(cnt, src), qtot = 0, qend = 0;
        double qD = 1.0;
        uint32_t qhash = REC ? (uint32_t)__shfl((int)hash, src) : 0u;
        const int bcbit = 2 * a + (neg ? 0 : 1);           // the boundary this axis runs into
        const bool per = (P.bc_periodic >> bcbit) & 1;
        const int qn = ax3 ? 0x7FFFFFFF : L[a], qmaxs = L[6];
        const int fb = L[3 + (ax3 ? 0 : a)] + (neg ? 0 : 1), ob = L[11 + (ax3 ? 0 : a)];   // exit face, offset of cell 0
        const int qstride = a == 0 ? 1 : (a == 1 ? L[0] : (a == 2 ? L[0] * L[1] : 0));
        gfloat* qT = lev_T(L);
        // (lane 3 is never the nearest face: distance 3e38)
        double qf = ax3 ? 3.0e38 : (double)s_face[fb + qc];
        while (__ballot(run)) {
            int lim = run ? min(kDrain, qmaxs - qcnt) : 0;
            int wall = -1;
            // a frozen quad (no ray, or its ray hit a wall inside the batch) has
            // length-0 crossings and does not move
            unsigned long long live = __ballot(run);
            int nlive = __popcll(live) >> 2;
            qs = run ? qs : 0.0;
            qi = run ? qi : 0.0;
            double dso[kDrain / 4];                        // crossing 4 k + a on lane a
            int oid[kDrain / 4], lin[kDrain / 4];
            // the two faces behind the exit face (a word past the axis's faces is
            // one of its LDS neighbours and is not used)
            double g = (double)s_face[fb + qc + st];
            float h = s_face[fb + qc + 2 * st];
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                int ov[4];
                oid[k] = lin[k] = 0;
                dso[k] = 0.0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int u = 4 * k + j;
                    ov[j] = s_off[ob + qc];
                    const double d = (qf - qp) * qi;
                    const double ds = quad_min_d(d);
                    dso[k] = a == j ? ds : dso[k];
                    unsigned long long em = __ballot(d == ds) & live;
                    qp = __builtin_amdgcn_inverse_ballot_w64(em) ? qf : qp + ds * qs;
                    // of several axes at the same distance the last one moves
                    if (__builtin_expect(__popcll(em) != nlive, 0))
                        em &= ~((em >> 1) | ((em >> 2) & 0x1111111111111111ull));
                    const bool mv = __builtin_amdgcn_inverse_ballot_w64(em);
                    if (REC) {
                        const int l = quad_sum(qc * qstride);
                        lin[k] = a == j ? l : lin[k];
                    }
                    qc += mv ? st : 0;
                    qf = mv ? g : qf;
                    g = mv ? (double)h : g;
                    const bool out = (uint32_t)qc >= (uint32_t)qn;
                    if (__builtin_expect(__ballot(out) != 0ull, 0)) {
                        int wl = -1;
                        if (out) {
                            if (per) {
                                qc = neg ? qn - 1 : 0;
                                qp = (double)s_face[fb + qc - st];
                            } else {
                                wl = bcbit;
                                qc -= st;
                            }
                            qf = (double)s_face[fb + qc];
                            g = (double)s_face[fb + qc + st];
                        }
                        wl = quad_max(wl);
                        const bool hit = wl >= 0;
                        wall = hit && u < lim ? wl : wall;
                        lim = hit ? min(lim, u + 1) : lim;
                        qs = hit ? 0.0 : qs;
                        qi = hit ? 0.0 : qi;
                        live &= ~__ballot(hit);
                        nlive = __popcll(live) >> 2;
                    }
                    h = s_face[fb + qc + 2 * st];
                }
                // the cells' field offsets: crossing 4 k + j to lane j
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int ou = quad_sum(ax3 ? 0 : ov[j]);
                    oid[k] = a == j ? ou : oid[k];
                }
            }
            if (__ballot(run && lim < kDrain)) {           // a wall or the step cap inside the batch
#pragma unroll
                for (int k = 0; k < kDrain / 4; ++k) dso[k] = 4 * k + a < lim ? dso[k] : 0.0;
            }
            // the cells' temperatures and lookups; each crossing's optical depth
            double Tv[kDrain / 4], dt[kDrain / 4], ibv[kDrain / 4], tk[kDrain / 4], dg[kDrain / 4];
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) Tv[k] = (double)load_T(qT, oid[k]);
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                double kap;
                if (SPEC == kSpecGreyT4) {
                    kap = (double)P.kappa_grey;
                    ibv[k] = Tv[k] * Tv[k] * Tv[k] * Tv[k];
                } else {
                    lookup_f64(P, Tv[k], qbg, qband, &kap, &ibv[k]);
                }
                dt[k] = kap * dso[k];
            }
            // summed in crossing order (every lane of the quad), kept by the
            // crossing's lane
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                const double t0 = qtau + quad_d<0x00>(dt[k]), t1 = t0 + quad_d<0x55>(dt[k]);
                const double t2 = t1 + quad_d<0xAA>(dt[k]);
                qtau = t2 + quad_d<0xFF>(dt[k]);
                tk[k] = a == 0 ? t0 : (a == 1 ? t1 : (a == 2 ? t2 : qtau));
            }
            // transmissivities; the first crossing past the cut-off
            int first = kDrain;
            double before = qtra;   // transmissivity before this group of four
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                const bool cut = tk[k] >= tau_cut;
                const double e1 = exp(-tk[k]);
                const double e0 = quad_d<kQuadPrev>(e1);   // (every lane of the quad takes part)
                const double ep = a == 0 ? before : e0;
                dg[k] = cut ? ep : ep - e1;
                first = min(first, cut ? 4 * k + a : kDrain);
                before = quad_d<0xFF>(e1);
            }
            bool cutq = false;
            int taken = lim;
            if (__ballot(first < lim)) {
                first = quad_min_i(first);
                cutq = first < lim;
                taken = cutq ? first + 1 : lim;
#pragma unroll
                for (int k = 0; k < kDrain / 4; ++k) dg[k] = 4 * k + a < taken ? dg[k] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < kDrain / 4; ++k) {
                const double x = dg[k] * ibv[k];
                qG += quad_d<0x00>(x);
                qG += quad_d<0x55>(x);
                qG += quad_d<0xAA>(x);
                qG += quad_d<0xFF>(x);
            }
            if (REC) {
                const uint32_t lb = (uint32_t)(P.nlev - 1) << 28;
#pragma unroll
                for (int k = 0; k < kDrain / 4; ++k) {
                    const uint32_t l0 = (uint32_t)quad_i<0x00>(lin[k]), l1 = (uint32_t)quad_i<0x55>(lin[k]);
                    const uint32_t l2 = (uint32_t)quad_i<0xAA>(lin[k]), l3 = (uint32_t)quad_i<0xFF>(lin[k]);
                    if (4 * k < taken) qhash = (qhash ^ (lb ^ l0)) * 16777619u;
                    if (4 * k + 1 < taken) qhash = (qhash ^ (lb ^ l1)) * 16777619u;
                    if (4 * k + 2 < taken) qhash = (qhash ^ (lb ^ l2)) * 16777619u;
                    if (4 * k + 3 < taken) qhash = (qhash ^ (lb ^ l3)) * 16777619u;
                }
            }
            qtra = before;   // (not used after a cut-off)
            qcnt += taken;
            qtot += taken;
            const bool hitw = run && !cutq && wall >= 0;
            if (hitw) qG += qtra * (double)s_ibw[wall * P.nB + qband];
            if (run && (cutq || hitw)) {
                run = false;
                qend = cutq ? 0 : 1;
                qtau = 0.0;   // (the quad idles below the cut-off: it adds 0)
                qtra = 1.0;
            } else if (run && qcnt >= qmaxs) {
                run = false;
                qend = 2;
                qD = 1.0 - qtra;
                qtau = 0.0;
                qtra = 1.0;
            }
        }
        // back to the lanes that held the rays
        const int from = alive ? 4 * rank : lane;
        const double rG = __shfl(qG, from), rD = __shfl(qD, from);
        const int rtot = __shfl(qtot, from), ren = __shfl(qend, from);
        const uint32_t rh = REC ? (uint32_t)__shfl((int)qhash, from) : 0u;
        if (alive) {
            G = rG;
            steps += rtot;
            if (REC) hash = rh;
            finish(rD, ren);
        }
        __builtin_amdgcn_s_setprio(0);
    }
    count_steps();
}
#define DN_TRACE64_INST(S, R, D) template __global__ void trace_f64<S, R, D>(TraceArgs, double2*);
#define DN_TRACE64_INST2(S, R) DN_TRACE64_INST(S, R, false) DN_TRACE64_INST(S, R, true)
DN_TRACE64_INST(kSpecTable, false, true)
DN_TRACE64_INST(kSpecTable, true, true)
DN_TRACE64_INST2(kSpecGreyT4, false)
DN_TRACE64_INST2(kSpecGreyT4, true)

#define DN_TRACE_INST(S, I, T, R, A, G) template __global__ void trace<S, I, T, R, A, G>(TraceArgs);
#define DN_TRACE_INST2(S, I, T, R, G) DN_TRACE_INST(S, I, T, R, false, G) DN_TRACE_INST(S, I, T, R, true, G)
#define DN_TRACE_INST3(S, I) DN_TRACE_INST2(S, I, 0, false, 0) DN_TRACE_INST2(S, I, 0, true, 0) \
    DN_TRACE_INST2(S, I, 1, false, 0) DN_TRACE_INST2(S, I, 0, false, 1) DN_TRACE_INST2(S, I, 0, false, 2)
DN_TRACE_INST3(kSpecTable, kTabSliced)
DN_TRACE_INST3(kSpecTable, kTabIbLds)
DN_TRACE_INST3(kSpecTable, kTabGlobal)
DN_TRACE_INST3(kSpecGreyT4, kTabGlobal)

// Range of the bricked level fields as order-preserving keys of their FP32
// values.  A wave takes a brick (64 cells) per load; one pair of atomics per
// block and level that has bricks for it (a wave's pair each, on the two words
// of a level, serialised at 11 ns: 376 us per level of 4.2e6 cells, now
// 27 us for that level and four coarser ones, 37 us for 25e6 cells).
__global__ __launch_bounds__(1024) void t_range(RangeArgs a)
{
    __shared__ unsigned s_lo[16], s_hi[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int w = blockIdx.x * 16 + wv, nw = gridDim.x * 16;
    const int x = ((lane >> 5) << 1) | (lane & 1), y = (lane >> 1) & 3, z = (lane >> 3) & 3;   // brick_index
    for (int l = 0; l < a.nlev; ++l) {
        const RangeLevel& L = a.lv[l];
        if ((int)blockIdx.x * 16 >= L.nbricks) continue;
        unsigned lo = 0xFFFFFFFFu, hi = 0u;
        for (int b0 = w; b0 < L.nbricks; b0 += 8 * nw) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = L.T[(size_t)min(b0 + u * nw, L.nbricks - 1) * 64 + lane];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const uint32_t b = (uint32_t)min(b0 + u * nw, L.nbricks - 1);
                const uint32_t r = fdiv(b, L.fd_nbx), bx = b - r * L.fd_nbx.d;
                const uint32_t bz = fdiv(r, L.fd_nby), by = r - bz * L.fd_nby.d;
                const unsigned k = __float_as_uint(v[u]);
                const unsigned key = (k & 0x80000000u) ? ~k : (k | 0x80000000u);
                if ((int)bx * 4 + x < L.n[0] && (int)by * 4 + y < L.n[1] && (int)bz * 4 + z < L.n[2]) {
                    lo = key < lo ? key : lo;
                    hi = key > hi ? key : hi;
                }
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            lo = min(lo, (unsigned)__shfl_xor((int)lo, off));
            hi = max(hi, (unsigned)__shfl_xor((int)hi, off));
        }
        if (lane == 0) {
            s_lo[wv] = lo;
            s_hi[wv] = hi;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int i = 1; i < 16; ++i) {
                lo = min(lo, s_lo[i]);
                hi = max(hi, s_hi[i]);
            }
            atomicMin(&a.keys[2 * l], lo);
            atomicMin(&a.keys[2 * l + 1], ~hi);
        }
        __syncthreads();
    }
}

// ------------------------------------------------------ reduce_rays ----
// Deterministic tallies: processing slot s owns rays [s*R, (s+1)*R) of the
// batch; their (E, A) are summed in ray order in FP64, Kahan-compensated FP32
// or plain FP32, and added to the slot's tally.  V: float2, or double2 of the
// FP64 traversal.
//
// A block takes NS slots, 1024 rays at a time through LDS (the next 1024 in
// flight), and a thread per slot adds its rays in order.  A slot's chain of
// additions is the bound where slots are few: NS = 16 there (the host's rule).
// 8192 rays for each of 1024 slots (double2, 134 MB): 1.16 ms with a thread per
// slot reading its rays from memory, 0.20 ms so; the chain alone is about 0.1.
template <typename V, int NS>
__global__ __launch_bounds__(256) void reduce_rays(const V* pray, int tally, long long nslots, int R, long long slot0,
                                                   const int4* slotinfo, double* E, double* A, double* Q2)
{
    constexpr int TR = 1024 / NS;                  // rays of a slot per tile
    __shared__ V tile[2][NS * (TR + 1)];
    const long long s0 = blockIdx.x * (long long)NS;
    const int ns = (int)min((long long)NS, nslots - s0);
    const int tid = threadIdx.x;
    V v[4];
    auto load = [&](long long r0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = tid + 256 * i, s = e / TR;
            const long long r = r0 + e % TR;
            v[i] = s < ns && r < R ? pray[(s0 + s) * R + r] : V{0, 0};
        }
    };
    auto put = [&](int b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = tid + 256 * i;
            tile[b][(e / TR) * (TR + 1) + e % TR] = v[i];
        }
    };
    double e = 0, a = 0, q = 0;
    float fe = 0, fa = 0, fq = 0, ce = 0, ca = 0, cq = 0;
    load(0);
    put(0);
    int b = 0;
    for (long long r0 = 0; r0 < R; r0 += TR, b ^= 1) {
        __syncthreads();
        load(r0 + TR);
        if (tid < ns) {
            const V* p = tile[b] + tid * (TR + 1);
            const int m = (int)min((long long)TR, R - r0);
            if (tally == DNSMC_TALLY_KAHAN_F32) {
#pragma unroll 4
                for (int r = 0; r < m; ++r) {
                    const float pe = (float)p[r].x, pa = (float)p[r].y;
                    float x = pe - pa;
                    float y = pe - ce, t = fe + y; ce = (t - fe) - y; fe = t;
                    y = pa - ca; t = fa + y; ca = (t - fa) - y; fa = t;
                    y = x * x - cq; t = fq + y; cq = (t - fq) - y; fq = t;
                }
            } else if (tally == DNSMC_TALLY_F32) {
#pragma unroll 4
                for (int r = 0; r < m; ++r) {
                    const float pe = (float)p[r].x, pa = (float)p[r].y;
                    float x = pe - pa;
                    fe += pe; fa += pa; fq += x * x;
                }
            } else {
#pragma unroll 8
                for (int r = 0; r < m; ++r) {
                    const double de = (double)p[r].x, da = (double)p[r].y, x = de - da;
                    e += de; a += da; q += x * x;
                }
            }
        }
        put(b ^ 1);
    }
    if (tid < ns) {
        const long long ts = slotinfo[slot0 + s0 + tid].x;
        const bool f32 = tally == DNSMC_TALLY_KAHAN_F32 || tally == DNSMC_TALLY_F32;
        E[ts] += f32 ? (double)fe : e;
        A[ts] += f32 ? (double)fa : a;
        Q2[ts] += f32 ? (double)fq : q;
    }
}
#define DN_REDUCE_INST(V, NS) template __global__ void reduce_rays<V, NS>(const V*, int, long long, int, long long, \
                                                                         const int4*, double*, double*, double*);
DN_REDUCE_INST(float2, 16)
DN_REDUCE_INST(float2, 64)
DN_REDUCE_INST(double2, 16)
DN_REDUCE_INST(double2, 64)

// ------------------------------------------------------------ finalize ----
// compat: nvar block estimates De_v = E_v - A_v; Q = mean; reference variance
// sum (De_v - Q)^2 / ((n - 0.5)(n - 1)) (code/mc_gpu.cu:217-222), sdev = sqrt.
// plain: Q = E - A, var(Q) = (R sum x^2 - Q^2)/(R - 1) from per-ray x = e - a.
// Eo and Ao (the mean emitted and absorbed parts) may be null.
__global__ void finalize(const double* E, const double* A, const double* Q2, long long nemit, int spe, int R,
                         int compat, double* Q, double* Eo, double* Ao, double* sd)
{
    long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (e >= nemit) return;
    if (compat) {
        double m = 0, me = 0, ma = 0;
        for (int v = 0; v < spe; ++v) {
            m += E[e * spe + v] - A[e * spe + v];
            me += E[e * spe + v];
            ma += A[e * spe + v];
        }
        m /= spe; me /= spe; ma /= spe;
        double var = 0;
        for (int v = 0; v < spe; ++v) {
            double d = (E[e * spe + v] - A[e * spe + v]) - m;
            var += 1.0 / (spe - 0.5) * 1.0 / (spe - 1) * d * d;
        }
        Q[e] = m; sd[e] = sqrt(var);
        if (Eo) Eo[e] = me;
        if (Ao) Ao[e] = ma;
    } else {
        double q = E[e] - A[e];
        double v = R > 1 ? ((double)R * Q2[e] - q * q) / (double)(R - 1) : 0.0;
        Q[e] = q; sd[e] = sqrt(v > 0 ? v : 0.0);
        if (Eo) Eo[e] = E[e];
        if (Ao) Ao[e] = A[e];
    }
}

// --------------------------------------------------------- spline pass ----
// One lane per grid line: natural-spline second derivatives through the fine
// values (forward sweep + back substitution, FP64), then evaluation at the
// coarse centres.  The grid-only factors come precomputed from the host.  The x
// pass sweeps the bricked fine field's lines once and evaluates every level on
// them (line j + n1 k); the y and z passes hold every level's lines (i + m0 k,
// i + m0 j) in one launch, and z writes the bricked layout of the levels.
//
// A sweep is one dependent chain per line, and the lines are few (a wave per CU
// on 256x128x128 cells), so what counts is that no load stands in the chain: the
// next kSpl values are in flight while a group is computed, the second
// derivatives lie [i][line] (whole lines per wave), the factors in LDS, and the
// x pass's rows leave through LDS in pieces of 16.  Five levels of 256x128x128
// cells: 12 launches of 128 us each (a load, a line-strided store and a
// coefficient load behind each other in the chain) -> 190 + 52 + 52 us.
constexpr int kSpl = 16;
template <int AXIS>
__global__ __launch_bounds__(64) void spline_pass(SplinePass s)
{
    extern __shared__ __align__(16) double s_f[];   // [6][nf] factors; x: 64 x 17 floats
    const int nf = s.nf, lane = threadIdx.x;
    double *f_ihh = s_f, *f_ihl = s_f + nf, *f_c6 = s_f + 2 * nf, *f_sig = s_f + 3 * nf, *f_invp = s_f + 4 * nf, *f_y2f = s_f + 5 * nf;
    float* s_t = (float*)(s_f + 6 * nf);
    for (int i = lane; i < nf; i += 64) {
        f_ihh[i] = s.ihh[i];
        f_ihl[i] = s.ihl[i];
        f_c6[i] = s.c6[i];
        f_sig[i] = s.sig[i];
        f_invp[i] = s.invp[i];
        f_y2f[i] = s.y2f[i];
    }
    int lv = 0, blk = blockIdx.x;
    if (AXIS != 0)
        for (int nb = (s.lv[0].nlines + 63) / 64; blk >= nb; nb = (s.lv[lv].nlines + 63) / 64) {
            blk -= nb;
            ++lv;
        }
    const SplineLevel& L0 = s.lv[lv];
    const int nl = L0.nlines, l = blk * 64 + lane, lc = min(l, nl - 1);   // (lanes past the last line repeat it)
    const bool live = l < nl;
    const float* in;
    long long st_in = 0;
    if (AXIS == 0) {
        in = s.fine + brick_index(0, lc % s.fn1, lc / s.fn1, s.fnbx, s.fnby);
    } else if (AXIS == 1) {
        in = L0.in + (lc % L0.m0) + (long long)(lc / L0.m0) * L0.m0 * s.fn1;
        st_in = L0.m0;
    } else {
        in = L0.in + lc;
        st_in = (long long)L0.m0 * L0.m1;
    }
    auto rd = [&](int i) -> float {
        return AXIS == 0 ? in[(size_t)(((i >> 2) << 6) | (((i >> 1) & 1) << 5) | (i & 1))] : in[(long long)i * st_in];
    };
    double* __restrict__ u = s.work + L0.work0 + lc;
    __syncthreads();
    float yn[kSpl];
    {   // forward
        double ym = (double)rd(0), y0 = (double)rd(min(1, nf - 1)), up = 0.0;
#pragma unroll
        for (int b = 0; b < kSpl; ++b) yn[b] = rd(min(2 + b, nf - 1));
        if (live) u[0] = 0.0;
        for (int i = 1; i < nf - 1; i += kSpl) {
            float yc[kSpl];
#pragma unroll
            for (int b = 0; b < kSpl; ++b) {
                yc[b] = yn[b];
                yn[b] = rd(min(i + kSpl + 1 + b, nf - 1));
            }
#pragma unroll
            for (int b = 0; b < kSpl; ++b) {
                if (i + b >= nf - 1) break;
                const double yp = (double)yc[b];
                const double dd = (yp - y0) * f_ihh[i + b] - (y0 - ym) * f_ihl[i + b];
                up = (f_c6[i + b] * dd - f_sig[i + b] * up) * f_invp[i + b];
                if (live) u[(size_t)(i + b) * nl] = up;
                ym = y0;
                y0 = yp;
            }
        }
        if (live) u[(size_t)(nf - 1) * nl] = 0.0;
    }
    {   // back
        double un = 0.0, vn[kSpl];
#pragma unroll
        for (int b = 0; b < kSpl; ++b) vn[b] = u[(size_t)max(nf - 2 - b, 0) * nl];
        for (int k = nf - 2; k >= 1; k -= kSpl) {
            double vc[kSpl];
#pragma unroll
            for (int b = 0; b < kSpl; ++b) {
                vc[b] = vn[b];
                vn[b] = u[(size_t)max(k - kSpl - b, 0) * nl];
            }
#pragma unroll
            for (int b = 0; b < kSpl; ++b) {
                if (k - b < 1) break;
                un = f_y2f[k - b] * un + vc[b];
                if (live) u[(size_t)(k - b) * nl] = un;
            }
        }
    }
    // evaluation
    constexpr int E = 8;
    for (int v = lv; v < (AXIS == 0 ? s.nlev : lv + 1); ++v) {
        const SplineLevel& L = s.lv[v];
        for (int q0 = 0; q0 < L.nc; q0 += 16) {
#pragma unroll
            for (int h = 0; h < 16; h += E) {
                float ya[E], yb[E];
                double ua[E], ub[E];
#pragma unroll
                for (int b = 0; b < E; ++b) {
                    const int k = L.klo[min(q0 + h + b, L.nc - 1)];
                    ya[b] = rd(k);
                    yb[b] = rd(k + 1);
                    ua[b] = u[(size_t)k * nl];
                    ub[b] = u[(size_t)(k + 1) * nl];
                }
#pragma unroll
                for (int b = 0; b < E; ++b) {
                    const int q = q0 + h + b;
                    if (q >= L.nc) break;
                    const double val = L.ca[q] * (double)ya[b] + L.cb[q] * (double)yb[b] + L.cA[q] * ua[b] + L.cB[q] * ub[b];
                    if (AXIS == 0) s_t[lane * 17 + h + b] = (float)val;
                    else if (!live) continue;
                    else if (AXIS == 1) L.out[(l % L.m0) + (long long)(l / L.m0) * L.m0 * L.m1 + (long long)q * L.m0] = (float)val;
                    else L.out[brick_index(l % L.m0, l / L.m0, q, L.nbx, L.nby)] = (float)val;
                }
            }
            if (AXIS == 0) {   // 64 rows of 16
                __syncthreads();
#pragma unroll
                for (int e = lane; e < 64 * 16; e += 64) {
                    const int r = e >> 4, q = q0 + (e & 15);
                    if (q < L.nc && blk * 64 + r < nl) L.out[(size_t)(blk * 64 + r) * L.nc + q] = s_t[r * 17 + (e & 15)];
                }
                __syncthreads();
            }
        }
    }
}
template __global__ void spline_pass<0>(SplinePass);
template __global__ void spline_pass<1>(SplinePass);
template __global__ void spline_pass<2>(SplinePass);

// Plain streaming copy (16 B per thread and iteration); the reference point
// for calibrating HBM byte counters.
__global__ void copy_f32x4(const float4* __restrict__ src, float4* __restrict__ dst, long long n4)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n4; i += (long long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// Streaming kernels of the achievable-bandwidth ceiling: every lane moves U
// 16-byte vectors per iteration (grid-stride, loads issued before stores),
// optionally with non-temporal hints.  stream_read sums what it reads and
// writes one float per thread only when the sum is the impossible value -1,
// so the loads are not removed and nothing else is written.
typedef float v4f __attribute__((ext_vector_type(4)));

template <int U, bool NT>
__global__ __launch_bounds__(256) void stream_copy(const float4* __restrict__ src4, float4* __restrict__ dst4,
                                                   long long n4)
{
    const v4f* src = (const v4f*)src4;
    v4f* dst = (v4f*)dst4;
    const long long st = (long long)gridDim.x * blockDim.x;
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    for (; i + (U - 1) * st < n4; i += U * st) {
        v4f v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = NT ? __builtin_nontemporal_load(src + i + u * st) : src[i + u * st];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (NT) __builtin_nontemporal_store(v[u], dst + i + u * st);
            else dst[i + u * st] = v[u];
        }
    }
    for (; i < n4; i += st) dst[i] = src[i];
}

template <int U, bool NT>
__global__ __launch_bounds__(256) void stream_read(const float4* __restrict__ src4, long long n4, float* sink)
{
    const v4f* src = (const v4f*)src4;
    const long long st = (long long)gridDim.x * blockDim.x;
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    float acc = 0.f;
    for (; i + (U - 1) * st < n4; i += U * st) {
        v4f v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = NT ? __builtin_nontemporal_load(src + i + u * st) : src[i + u * st];
#pragma unroll
        for (int u = 0; u < U; ++u) acc += (v[u].x + v[u].y) + (v[u].z + v[u].w);
    }
    for (; i < n4; i += st) acc += src[i].x;
    if (acc == -1.0f) sink[blockIdx.x * (long long)blockDim.x + threadIdx.x] = acc;
}

template __global__ void stream_copy<1, false>(const float4*, float4*, long long);
template __global__ void stream_copy<4, false>(const float4*, float4*, long long);
template __global__ void stream_copy<4, true>(const float4*, float4*, long long);
template __global__ void stream_read<1, false>(const float4*, long long, float*);
template __global__ void stream_read<4, false>(const float4*, long long, float*);
template __global__ void stream_read<4, true>(const float4*, long long, float*);

// ------------------------------------------------- DNS coupling slabs ----
// fix_temp (code/fix_var.f:49-73) for one rank's slab, written straight into
// the bricked device field instead of summed into a full-size host buffer and
// all-reduced: T(i,j,k) = cnew * Tc / Tplus + Tc in FP64 (left to right, as
// the Fortran expression), rounded to FP32 as the real(4) TMC is.  cnew is the
// rank's array cnew(0:n0+1, nj, nk), i fastest; global (i, j, k) of the slab
// (1-based, i0..i0+ni-1 etc.) reads cnew(i - i0 + 1, j - j0 + 1, k - k0 + 1).
// Ghost indices (0 and n+1) are not part of the bricked field and are skipped.
__global__ void slab_to_field(const double* cnew, int n0, int n1, int n2, int i0, int j0, int k0, int ni, int nj,
                              int nk, double Tc, double Tplus, float* T, int nbx, int nby)
{
    const long long n = (long long)ni * nj * nk;
    for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n; c += (long long)gridDim.x * blockDim.x) {
        const int a = (int)(c % ni), b = (int)((c / ni) % nj), d = (int)(c / ((long long)ni * nj));
        const int i = i0 + a, j = j0 + b, k = k0 + d;
        if (i < 1 || i > n0 || j < 1 || j > n1 || k < 1 || k > n2) continue;
        const double v = cnew[(long long)(a + 1) + (long long)(n0 + 2) * (b + (long long)nj * d)];
        T[brick_index(i - 1, j - 1, k - 1, nbx, nby)] = (float)(v * Tc / Tplus + Tc);
    }
}

// get_results_ (code/mc_gpu.cu:759-776): Q and its standard error of the
// emitters in the j slab [jlo, jlo + nj) (0-based) into real(4) arrays
// (0:n0+1, 0:nj+1, 0:n2+1), i fastest; other entries keep their values.
__global__ void results_to_fortran(const int* emit, long long nemit, const double* Q, const double* sd, int n0,
                                   int n1, int jlo, int nj, int n2, float* resf, float* varf)
{
    const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (e >= nemit) return;
    const int cell = emit[e];
    const int i = cell % n0, j = (cell / n0) % n1, k = cell / (n0 * n1);
    const int jl = j - jlo;
    if (jl < 0 || jl >= nj || k >= n2) return;
    const long long o = (long long)(i + 1) + (long long)(n0 + 2) * ((jl + 1) + (long long)(nj + 2) * (k + 1));
    resf[o] = (float)Q[e];
    varf[o] = (float)sd[e];
}

// The same where every interior entry has a result, in row order: [Q | standard
// error] as FP32, for the host to place.
__global__ void results_to_f32(const double* Q, const double* sd, long long n, float* out)
{
    const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (e >= n) return;
    out[e] = (float)Q[e];
    out[n + e] = (float)sd[e];
}

// fix_rad (code/fix_var.f:75-121) for one rank's k range, from the device
// results: divQ(i, jl, k - k0 + 1) = Q / stefan / Tc^4 and vcore likewise from
// the standard error, for the emitters in the solver's j slab [jlo, jlo + nj)
// (0-based) and k in [k0, k0 + nk) (0-based); out arrays (0:n0+1, nj, nk).
__global__ void field_to_slab(const int* emit, long long nemit, const double* Q, const double* sd, int n0, int n1,
                              int jlo, int nj, int k0, int nk, double stefan, double tc4, double* divq, double* vcore)
{
    const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (e >= nemit) return;
    const int cell = emit[e];
    const int i = cell % n0, j = (cell / n0) % n1, k = cell / (n0 * n1);
    const int jl = j - jlo, kl = k - k0;
    if (jl < 0 || jl >= nj || kl < 0 || kl >= nk) return;
    const long long o = (long long)(i + 1) + (long long)(n0 + 2) * (jl + (long long)nj * kl);
    divq[o] = Q[e] / stefan / tc4;
    vcore[o] = sd[e] / stefan / tc4;
}

// A temperature field in the reference's layout, T(0:n0+1, 0:n1+1, 0:n2+1) with
// i fastest (code/param.h:104-105), into the 4x4x4-bricked layout: interior
// cells only (the ghost layers are not part of the bricked field).
__global__ void ghost_to_bricks(const float* Tg, int n0, int n1, int n2, float* T, int nbx, int nby)
{
    const long long n = (long long)n0 * n1 * n2;
    for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n; c += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(c % n0), j = (int)((c / n0) % n1), k = (int)(c / ((long long)n0 * n1));
        T[brick_index(i, j, k, nbx, nby)] = Tg[(long long)(i + 1) + (long long)(n0 + 2) * ((j + 1) + (long long)(n1 + 2) * (k + 1))];
    }
}

// Table-coordinate field of the sliced-table traversal: u = clamp(T/dT - T0/dT,
// 0, nT-1) - lo, the position of each cell's temperature among the nodes held
// in LDS.  The traversal's lerp from u is bit-identical to the one from T (the
// subtraction of the integer lo from the clamped position is exact).
__global__ void t_to_u(const float* T, float* U, long long n, float inv_dT, float mT0, float top, float lo)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        float pos = fmaf(T[i], inv_dT, mT0);
        pos = fminf(fmaxf(pos, 0.0f), top);
        U[i] = pos - lo;
    }
}

__global__ void fill_u32(unsigned* p, long long n, unsigned v)
{
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// A run's start: the tallies and the two step counters, one launch (four fills
// before; a solve of 2e5 rays waits for each launch).
__global__ void clear_tallies(double* E, double* A, double* Q2, long long n, unsigned long long* nsteps)
{
    const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (i < n) {
        E[i] = 0.0;
        A[i] = 0.0;
        Q2[i] = 0.0;
    }
    if (i < 2) nsteps[i] = 0ull;
}

__global__ void fill_f64(double* p, long long n, double v)
{
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

}  // namespace dn
