// Learned importance-sampling proposal (gfx950): BF16 MFMA forward/backward
// training kernels, the per-cell features, the training samples taken from a
// plain run, and the ray generator that samples from the network.
//
// No counterpart in the reference: its proposal is the fixed Tmax
// distribution (code/mc_gpu.cu:584-590, :830-896).  Every learned ray carries
// the factor p/q (plain over learned probability of its direction bin and
// (band, g) bin), so the estimator's mean is the plain estimator's mean; a
// defensive mixture q = (1 - eps) q_net + eps p bounds p/q by 1/eps.
//
// Matrix products use v_mfma_f32_16x16x16_bf16 (FP32 accumulate).  Operand
// layout of one 16x16x16 step for lane l (0..63), element i (0..3):
//   A(row = l % 16, k = 4 (l / 16) + i),  B(k = 4 (l / 16) + i, col = l % 16),
//   D(row = 4 (l / 16) + i, col = l % 16).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dmath.h"
#include "kernels.h"
#include "mlp.h"

namespace dn {

typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));


// Fragment of a 16-row panel starting at row r0, k-block k0: element (r, k)
// of the operand is M[r * rs + k * cs].
__device__ __forceinline__ s4v frag(const uint16_t* M, int rs, int cs, int r0, int k0, int lane)
{
    const int r = r0 + (lane & 15), k = k0 + 4 * (lane >> 4);
    const uint16_t* p = M + r * rs + k * cs;
    s4v v;
    if (cs == 1) {   // four consecutive BF16 (8-byte aligned): one LDS read
        const uint2 u = *(const uint2*)p;
        v.x = (short)(u.x & 0xFFFFu);
        v.y = (short)(u.x >> 16);
        v.z = (short)(u.y & 0xFFFFu);
        v.w = (short)(u.y >> 16);
        return v;
    }
    v.x = (short)p[0];
    v.y = (short)p[cs];
    v.z = (short)p[2 * cs];
    v.w = (short)p[3 * cs];
    return v;
}

// 64x64 output per 256-thread block (each wave a 32x32 quadrant of 2x2
// 16x16 tiles): acc += A[64 x K] B[K x 64], A(r, k) = A[r*ars + k*acs],
// B(k, n) = B[k*brs + n*bcs].  acc[ti][tj][i] holds element
// (row = qr + 16 ti + 4 (lane/16) + i, col = qc + 16 tj + lane % 16).
__device__ __forceinline__ void gemm64(const uint16_t* A, int ars, int acs, const uint16_t* B, int brs, int bcs, int K,
                                       f4v acc[2][2])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int qr = (w >> 1) * 32, qc = (w & 1) * 32;
    for (int k0 = 0; k0 < K; k0 += 16) {
        const s4v a0 = frag(A, ars, acs, qr, k0, lane), a1 = frag(A, ars, acs, qr + 16, k0, lane);
        const s4v b0 = frag(B, bcs, brs, qc, k0, lane), b1 = frag(B, bcs, brs, qc + 16, k0, lane);
        acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1, b1, acc[1][1], 0, 0, 0);
    }
}

__device__ __forceinline__ void acc_zero(f4v acc[2][2])
{
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) acc[a][b] = f4v{0.f, 0.f, 0.f, 0.f};
}

// Visit every accumulator element with its (row, col) in the 64x64 tile.
template <class F>
__device__ __forceinline__ void acc_each(const f4v acc[2][2], F f)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int qr = (w >> 1) * 32, qc = (w & 1) * 32;
    for (int ti = 0; ti < 2; ++ti)
        for (int tj = 0; tj < 2; ++tj)
            for (int i = 0; i < 4; ++i) f(qr + 16 * ti + 4 * (lane >> 4) + i, qc + 16 * tj + (lane & 15), acc[ti][tj][i]);
}

// H1 = tanh(X W1 + b1) for rows < nrow (zero rows after), BF16.
__device__ __forceinline__ void layer1(const float* sX, const MlpWeights& w, int nrow, uint16_t* H1b, int hs = kMlpHid)
{
    for (int e = threadIdx.x; e < 64 * kMlpHid; e += blockDim.x) {
        const int s = e / kMlpHid, j = e - s * kMlpHid;
        float h = 0.f;
        if (s < nrow) {
            float acc = w.b1[j];
            for (int i = 0; i < kMlpIn; ++i) acc = fmaf(sX[s * kMlpIn + i], bf2f(w.W1[i * kMlpHid + j]), acc);
            h = tanhf(acc);
        }
        H1b[s * hs + j] = f2bf(h);
    }
}

// Barrier for the block's LDS traffic only: each wave's LDS operations are
// complete before it, its global stores (the rows, read by no other thread
// of this kernel) stay in flight.
__device__ __forceinline__ void lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Tile jt of W3^T (rows jt*64 .. jt*64 + 63 of the [noutp][64] copy, 128 B
// each) for a 256-thread block in two steps: its two 16-byte pieces per
// thread into registers (issued one tile ahead), then into the padded LDS
// rows (8-byte writes: the padded rows are 8-byte aligned).
__device__ __forceinline__ void load_w3_tile(const uint16_t* W3T, int jt, uint4& r0, uint4& r1)
{
    const uint4* src = (const uint4*)(W3T + (size_t)jt * 64 * 64);
    r0 = src[threadIdx.x];
    r1 = src[threadIdx.x + 256];
}
__device__ __forceinline__ void put_w3_tile(const uint4& r0, const uint4& r1, uint16_t* dst)
{
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int e = (int)threadIdx.x + 256 * i, n = e >> 3, k8 = e & 7;
        const uint4 r = i ? r1 : r0;
        uint2* d = (uint2*)(dst + n * kPropStride + k8 * 8);
        d[0] = make_uint2(r.x, r.y);
        d[1] = make_uint2(r.z, r.w);
    }
}

// ------------------------------------------------------------- training ----
// One gradient evaluation, four launches over 64-row blocks of the minibatch:
//   mlp_train_prep  the sum of the sample weights; W3 with the input index
//                   contiguous (the logits' operand layout),
//   mlp_train_rows  per 64 rows (16 per wave): forward, log-sum-exp of both
//                   heads, dH2 and the gradients below W3; H2 and the rows'
//                   log-sum-exps to memory,
//   mlp_train_w3    per 64 columns of W3 and split of the rows: the logits and
//                   dZ again, dW3 and db3 summed over the split in registers,
//   mlp_reduce      the partial sums.
// The first form wrote every 64-row block's whole gradient (451 KB) and summed
// 256 of them: 115 MB each way, 0.42 ms per step of 16384 rows (320 us of tile
// kernel at one block per CU, 79 us of reduction, 19 us of weight sum).  Here
// W3's part (96 % of the parameters) is kept in registers over the rows of a
// split: 0.14 ms for the same step (462 -> 142 us with the update; kernels 73 us
// for the rows, a block per CU and so one wave per SIMD, bound by that wave's
// chain through two passes over W3's columns (VALU at 0.40 of its issue peak);
// 26 us for dW3, 11 us for the sums).  Every sum over rows, columns and blocks
// below W3 keeps the first form's order, so those gradients are bit for bit what
// they were.  dZ leaves the logits' accumulators in the layout of the next
// product's operand (rows 4 (l / 16) + i, column l % 16), so dW3 = H2^T dZ takes
// it from registers.

// Four BF16 of consecutive k as an MFMA operand, from an 8-byte aligned address.
__device__ __forceinline__ s4v frag8(const uint16_t* p)
{
    const uint2 u = *(const uint2*)p;
    s4v v;
    v.x = (short)(u.x & 0xFFFFu);
    v.y = (short)(u.x >> 16);
    v.z = (short)(u.y & 0xFFFFu);
    v.w = (short)(u.y >> 16);
    return v;
}
// Four FP32 as BF16, round to nearest even (v_cvt_pk_bf16_f32).
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 b2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ s4v pack4(float a, float b, float c, float d)
{
    const uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2v{a, b}, b2v));
    const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2v{c, d}, b2v));
    s4v v;
    v.x = (short)(lo & 0xFFFFu);
    v.y = (short)(lo >> 16);
    v.z = (short)(hi & 0xFFFFu);
    v.w = (short)(hi >> 16);
    return v;
}
__device__ __forceinline__ void put8(uint16_t* p, s4v v)
{
    *(uint2*)p = make_uint2((uint32_t)(uint16_t)v.x | ((uint32_t)(uint16_t)v.y << 16),
                            (uint32_t)(uint16_t)v.z | ((uint32_t)(uint16_t)v.w << 16));
}
#define DN_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0)

// dZ = w (softmax - onehot) of a logit z, its head's log-sum-exp and whether
// its column is the sample's bin.
__device__ __forceinline__ float mlp_dz(float z, float w, float lse, bool hot)
{
    return w * (__expf(z - lse) - (hot ? 1.f : 0.f));
}

// Block 0: wsum = sum of wt (per thread in steps of 256, eight loads in flight,
// then a tree).  Block 1 + jt: rows 64 jt .. 64 jt + 63 of W3T[noutp][64].
__global__ __launch_bounds__(256) void mlp_train_prep(const float* wt, long long n, float* wsum, const uint16_t* W3,
                                                      int noutp, uint16_t* W3T)
{
    __shared__ float s[256];
    __shared__ uint16_t t[64 * kPropStride];
    const int tid = threadIdx.x;
    if (blockIdx.x == 0) {
        float v = 0.f;
        long long i = tid;
        for (; i + 7 * 256 < n; i += 8 * 256) {
            float x[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) x[u] = wt[i + u * 256];
#pragma unroll
            for (int u = 0; u < 8; ++u) v += x[u];
        }
        for (; i < n; i += 256) v += wt[i];
        s[tid] = v;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o) s[tid] += s[tid + o];
            __syncthreads();
        }
        if (tid == 0) *wsum = s[0] > 0.f ? s[0] : 1.f;
        return;
    }
    const int jt = blockIdx.x - 1;
    for (int e = tid; e < 512; e += 256) {
        const int h = e >> 3, c8 = e & 7;
        const uint4 r = ((const uint4*)W3)[((size_t)h * noutp + jt * 64) / 8 + c8];
        uint2* d = (uint2*)(t + h * kPropStride + c8 * 8);
        d[0] = make_uint2(r.x, r.y);
        d[1] = make_uint2(r.z, r.w);
    }
    __syncthreads();
    for (int e = tid; e < 1024; e += 256) {
        const int c = e >> 4, h = (e & 15) * 4;
        s4v v;
        v.x = (short)t[h * kPropStride + c];
        v.y = (short)t[(h + 1) * kPropStride + c];
        v.z = (short)t[(h + 2) * kPropStride + c];
        v.w = (short)t[(h + 3) * kPropStride + c];
        put8(W3T + ((size_t)jt * 64 + c) * 64 + h, v);
    }
}

// Tile jt of row-major W3 (64 rows h, columns 64 jt .. + 63) in two steps, as
// load_w3_tile / put_w3_tile take W3T's.
__device__ __forceinline__ void load_w3_cols(const uint16_t* W3, int noutp, int jt, uint4& r0, uint4& r1)
{
    const uint4* src = (const uint4*)W3;
    const int e = threadIdx.x;
    r0 = src[((size_t)(e >> 3) * noutp + jt * 64) / 8 + (e & 7)];
    r1 = src[((size_t)((e >> 3) + 32) * noutp + jt * 64) / 8 + (e & 7)];
}

// One wave per 16 rows.  The logits are formed transposed, Z^T = W3^T H2^T: lane
// l holds sample l % 16 and columns 4 (l / 16) + i of a 16-column tile, which is
// the layout of dH2 = dZ W3^T's first operand, so dZ stays in registers.  Sums
// over the rows and the log-sum-exps (four chains of 16 columns per tile and
// row, merged at the end) run in a fixed order.
__global__ __launch_bounds__(256) void mlp_train_rows(MlpTrainArgs a)
{
    constexpr int PS = kPropStride;
    __shared__ __align__(16) uint16_t sA[2 * 64 * PS];   // W3^T tiles (two); H1 before; dA2 [row][col], H1^T [h][row] after
    __shared__ __align__(16) uint16_t sB[2 * 64 * PS];   // W3 tiles (two); W2 before; W2, dA2^T [col][row] after
    __shared__ __align__(16) float sZ[64 * PS];          // logits [row][col]; dA2, dA1 after
    __shared__ float sX[64 * kMlpIn];
    __shared__ float sl[64];
    __shared__ __align__(16) float slse[128];
    const int noutp = a.w.noutp, nbin = a.w.nbin, ntile = noutp / 64;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int lc = lane & 15, lr = 4 * (lane >> 4);    // this lane's column and first row of a 16 x 16 tile
    const int wr = 16 * wv;                            // the wave's first row
    const long long r0 = (long long)blockIdx.x * 64;
    const int nrow = (int)((a.n - r0) < 64 ? (a.n - r0) : 64);
    const float inv_w = 1.0f / *a.wsum;

    for (int e = tid; e < 64 * kMlpIn; e += 256) {
        const int s = e / kMlpIn;
        sX[e] = s < nrow ? a.X[(r0 + s) * kMlpIn + (e - s * kMlpIn)] : 0.f;
    }
    for (int e = tid; e < 4096; e += 256) sB[(e >> 6) * PS + (e & 63)] = a.w.W2[e];
    // this lane's sample (row wr + lc)
    const bool have = wr + lc < nrow;
    const float sw = have ? a.wt[r0 + wr + lc] * inv_w : 0.f;
    const int td = have ? a.td[r0 + wr + lc] : 0;
    const int tb = kMlpDir + (have ? a.tb[r0 + wr + lc] : 0);
    if (lr == 0) a.sw[r0 + wr + lc] = sw;
    __syncthreads();
    // H1 in the accumulators' layout: h1[4 tj + i] = H1(row lr + i, col 16 tj + lc)
    float h1[16], h2[16];
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) {
        const int j = 16 * tj + lc;
        float wj[kMlpIn];
#pragma unroll
        for (int i = 0; i < kMlpIn; ++i) wj[i] = bf2f(a.w.W1[i * kMlpHid + j]);
        const float bj = a.w.b1[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float acc = bj;
#pragma unroll
            for (int i = 0; i < kMlpIn; ++i) acc = fmaf(sX[(wr + lr + r) * kMlpIn + i], wj[i], acc);
            h1[4 * tj + r] = wr + lr + r < nrow ? tanhf(acc) : 0.f;
            sA[(wr + lr + r) * PS + j] = f2bf(h1[4 * tj + r]);
        }
    }
    __syncthreads();
    uint16_t* sH = sA + 64 * PS;   // H2 [row][h] (each wave its own rows)
    {   // H2 = tanh(H1 W2 + b2)
        f4v acc[4];
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) acc[tj] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < 64; k0 += 16) {
            const s4v av = frag8(sA + (wr + lc) * PS + k0 + lr);
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                const uint16_t* q = sB + (k0 + lr) * PS + 16 * tj + lc;
                s4v bv;
                bv.x = (short)q[0];
                bv.y = (short)q[PS];
                bv.z = (short)q[2 * PS];
                bv.w = (short)q[3 * PS];
                acc[tj] = DN_MFMA(av, bv, acc[tj]);
            }
        }
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) {
            const float bj = a.w.b2[16 * tj + lc];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float h = wr + lr + r < nrow ? tanhf(acc[tj][r] + bj) : 0.f;
                h2[4 * tj + r] = h;
                sH[(wr + lr + r) * PS + 16 * tj + lc] = f2bf(h);
            }
            // H2^T of the block, [h][row], for mlp_train_w3
            put8(a.H2T + ((size_t)blockIdx.x * 64 + 16 * tj + lc) * 64 + wr + lr,
                 pack4(h2[4 * tj], h2[4 * tj + 1], h2[4 * tj + 2], h2[4 * tj + 3]));
        }
    }
    lds_sync();
    s4v ha[4];   // H2 as an operand: row lc of the wave, h = 16 k + lr + i
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        ha[k] = frag8(sH + (wr + lc) * PS + 16 * k + lr);
        put8(a.H2 + (r0 + wr + lc) * 64 + 16 * k + lr, ha[k]);
    }
    lds_sync();  // (H1, W2 and H2 read: the tiles take their place)
    // b3 of this lane's columns of tile jt
    auto bias = [&](int jt, f4v* b) {
#pragma unroll
        for (int tj = 0; tj < 4; ++tj)
#pragma unroll
            for (int i = 0; i < 4; ++i) b[tj][i] = a.w.b3[jt * 64 + 16 * tj + lr + i];
    };
    // pass 1: log-sum-exp of both heads, online over the column tiles: thread
    // (row, part) over columns 16 part .. 16 part + 15, the four merged at the end
    float lse_d, lse_b;
    {
        const int row = tid >> 2, part = tid & 3;      // a row of this wave
        float m = -3.0e38f, sum = 0.f, zt = 0.f, md = 0.f, sd = 0.f, ztd = 0.f;
        const int rtd = __shfl(td, row & 15), rtb = __shfl(tb, row & 15);
        uint4 t0, t1;
        f4v b3[4];
        load_w3_tile(a.W3T, 0, t0, t1);
        bias(0, b3);
        put_w3_tile(t0, t1, sA);
        for (int jt = 0; jt < ntile; ++jt) {
            const uint16_t* sW = sA + (jt & 1) * 64 * PS;
            const int jn = min(jt + 1, ntile - 1);
            load_w3_tile(a.W3T, jn, t0, t1);
            lds_sync();
            f4v acc[4];
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) acc[tj] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int tj = 0; tj < 4; ++tj)
                    acc[tj] = DN_MFMA(frag8(sW + (16 * tj + lc) * PS + 16 * k + lr), ha[k], acc[tj]);
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) *(f4v*)(sZ + (wr + lc) * PS + 16 * tj + lr) = acc[tj] + b3[tj];
            bias(jn, b3);
            put_w3_tile(t0, t1, sA + ((jt + 1) & 1) * 64 * PS);
            if (jt == 1) {   // the (band, g) head starts
                md = m;
                sd = sum;
                ztd = zt;
                m = -3.0e38f;
                sum = zt = 0.f;
            }
            // (this wave's rows of sZ only)
            const int hot = (jt == 0 ? rtd : rtb) - jt * 64 - part * 16;
            const int nc = min(16, kMlpDir + nbin - jt * 64 - part * 16);   // columns of a head
            const float* zr = sZ + row * PS + part * 16;
            float z[16], mm[17], t[16];
            mm[0] = m;
#pragma unroll
            for (int c = 0; c < 16; ++c) z[c] = zr[c];
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                mm[c + 1] = c < nc ? fmaxf(mm[c], z[c]) : mm[c];
                if (c == hot) zt = z[c];
            }
#pragma unroll
            for (int c = 0; c < 16; ++c) t[c] = __expf(-fabsf(z[c] - mm[c]));
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                const float sn = z[c] > mm[c] ? sum * t[c] + 1.f : sum + t[c];
                sum = c < nc ? sn : sum;
            }
            m = mm[16];
        }
        for (int o = 1; o < 4; o <<= 1) {   // merge the four partial (max, sum) pairs of the row
            const float md2 = __shfl_xor(md, o, 4), sd2 = __shfl_xor(sd, o, 4);
            const float mb2 = __shfl_xor(m, o, 4), sb2 = __shfl_xor(sum, o, 4);
            const float mdn = fmaxf(md, md2), mbn = fmaxf(m, mb2);
            sd = sd * __expf(md - mdn) + sd2 * __expf(md2 - mdn);
            sum = sum * __expf(m - mbn) + sb2 * __expf(mb2 - mbn);
            md = mdn;
            m = mbn;
            ztd += __shfl_xor(ztd, o, 4);
            zt += __shfl_xor(zt, o, 4);
        }
        const float swr = __shfl(sw, row & 15);
        if (part == 0) {   // log-sum-exp per head; the sample's loss
            const float ld = md + __logf(sd), lb = m + __logf(sum);
            slse[2 * row] = ld;
            slse[2 * row + 1] = lb;
            a.lse[2 * (r0 + row)] = ld;
            a.lse[2 * (r0 + row) + 1] = lb;
            sl[row] = swr * ((ld - ztd) + (lb - zt));
        }
        lds_sync();
        lse_d = slse[2 * (wr + lc)];
        lse_b = slse[2 * (wr + lc) + 1];
    }
    // pass 2: dZ = w (softmax - onehot), dH2 = dZ W3^T
    f4v dh[4];
#pragma unroll
    for (int th = 0; th < 4; ++th) dh[th] = f4v{0.f, 0.f, 0.f, 0.f};
    {
        uint4 t0, t1, c0, c1;
        f4v b3[4];
        load_w3_tile(a.W3T, 0, t0, t1);
        load_w3_cols(a.w.W3, noutp, 0, c0, c1);
        bias(0, b3);
        put_w3_tile(t0, t1, sA);
        put_w3_tile(c0, c1, sB);
        for (int jt = 0; jt < ntile; ++jt) {
            const uint16_t* sW = sA + (jt & 1) * 64 * PS;
            const uint16_t* sC = sB + (jt & 1) * 64 * PS;
            const int jn = min(jt + 1, ntile - 1);
            load_w3_tile(a.W3T, jn, t0, t1);
            load_w3_cols(a.w.W3, noutp, jn, c0, c1);
            lds_sync();
            f4v acc[4];
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) acc[tj] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int tj = 0; tj < 4; ++tj)
                    acc[tj] = DN_MFMA(frag8(sW + (16 * tj + lc) * PS + 16 * k + lr), ha[k], acc[tj]);
            const float lse = jt == 0 ? lse_d : lse_b;
            const int hot = (jt == 0 ? td : tb) - jt * 64 - lr, nc = kMlpDir + nbin - jt * 64 - lr;
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                float dz[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = mlp_dz(acc[tj][i] + b3[tj][i], sw, lse, hot == 16 * tj + i);
                    dz[i] = 16 * tj + i < nc ? v : 0.f;
                }
                const s4v dv = pack4(dz[0], dz[1], dz[2], dz[3]);
#pragma unroll
                for (int th = 0; th < 4; ++th)
                    dh[th] = DN_MFMA(dv, frag8(sC + (16 * th + lc) * PS + 16 * tj + lr), dh[th]);
            }
            bias(jn, b3);
            put_w3_tile(t0, t1, sA + ((jt + 1) & 1) * 64 * PS);
            put_w3_tile(c0, c1, sB + ((jt + 1) & 1) * 64 * PS);
        }
    }
    __syncthreads();
    // layer 2 backward: dA2 = dH2 (1 - H2^2); W2 again
    uint16_t *sD = sA, *sHT = sA + 64 * PS, *sW2 = sB, *sDT = sB + 64 * PS;   // dA2, H1^T, W2, dA2^T
    for (int e = tid; e < 4096; e += 256) sW2[(e >> 6) * PS + (e & 63)] = a.w.W2[e];
    float* part = a.part + (size_t)blockIdx.x * kMlpSmall;
    const MlpLayout L = mlp_layout(nbin);
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) {
        float d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float h = h2[4 * tj + i];
            d[i] = dh[tj][i] * (1.f - h * h);
            sZ[(wr + lr + i) * PS + 16 * tj + lc] = d[i];
            sD[(wr + lr + i) * PS + 16 * tj + lc] = f2bf(d[i]);
        }
        put8(sDT + (16 * tj + lc) * PS + wr + lr, pack4(d[0], d[1], d[2], d[3]));
        put8(sHT + (16 * tj + lc) * PS + wr + lr, pack4(h1[4 * tj], h1[4 * tj + 1], h1[4 * tj + 2], h1[4 * tj + 3]));
    }
    __syncthreads();
    if (tid < 64) {
        float s = 0.f;
        for (int r = 0; r < 64; ++r) s += sZ[r * PS + tid];
        part[L.ob2 + tid] = s;
    }
    {   // dW2 = H1^T dA2: this wave's 16 rows h
        f4v acc[4];
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) acc[tj] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < 64; k0 += 16) {
            const s4v av = frag8(sHT + (wr + lc) * PS + k0 + lr);
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) acc[tj] = DN_MFMA(av, frag8(sDT + (16 * tj + lc) * PS + k0 + lr), acc[tj]);
        }
#pragma unroll
        for (int tj = 0; tj < 4; ++tj)
#pragma unroll
            for (int i = 0; i < 4; ++i) part[L.oW2 + (wr + lr + i) * 64 + 16 * tj + lc] = acc[tj][i];
    }
    {   // dA1 = (dA2 W2^T)(1 - H1^2)
        f4v acc[4];
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) acc[tj] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < 64; k0 += 16) {
            const s4v av = frag8(sD + (wr + lc) * PS + k0 + lr);
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) acc[tj] = DN_MFMA(av, frag8(sW2 + (16 * tj + lc) * PS + k0 + lr), acc[tj]);
        }
        __syncthreads();   // db2's sums have read sZ
#pragma unroll
        for (int tj = 0; tj < 4; ++tj)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float h = h1[4 * tj + i];
                sZ[(wr + lr + i) * PS + 16 * tj + lc] = acc[tj][i] * (1.f - h * h);
            }
    }
    __syncthreads();
    for (int e = tid; e < (kMlpIn + 1) * kMlpHid; e += 256) {   // dW1 = X^T dA1 (FP32), db1
        const int i = e >> 6, j = e & 63;
        float s = 0.f;
        if (i < kMlpIn) {
            for (int r = 0; r < 64; ++r) s = fmaf(sX[r * kMlpIn + i], sZ[r * PS + j], s);
        } else {
            for (int r = 0; r < 64; ++r) s += sZ[r * PS + j];
        }
        part[(i < kMlpIn ? L.oW1 + i * kMlpHid : L.ob1) + j] = s;
    }
    if (tid == 192) {
        float s = 0.f;
        for (int r = 0; r < 64; ++r) s += sl[r];
        a.loss_part[blockIdx.x] = s;
    }
}

// dW3 and db3 of column tile jt = blockIdx.x over the 64-row blocks of split
// blockIdx.y; wave w holds columns 16 w .. 16 w + 15.
__global__ __launch_bounds__(256) void mlp_train_w3(MlpTrainArgs a, int per)
{
    constexpr int PS = kPropStride;
    __shared__ __align__(16) uint16_t sH[2][64 * PS], sHT[2][64 * PS];   // H2 [row][h], H2^T [h][row]
    __shared__ __align__(16) float slse[2][64], ssw[2][64];
    __shared__ __align__(16) int shot[2][64];
    const int noutp = a.w.noutp, jt = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int lc = lane & 15, lr = 4 * (lane >> 4);
    const int col = jt * 64 + 16 * wv + lc;
    const bool used = col < kMlpDir + a.w.nbin;
    const long long nblk = (a.n + 63) / 64;
    const long long b0 = (long long)blockIdx.y * per, b1 = b0 + per < nblk ? b0 + per : nblk;
    s4v wf[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) wf[k] = frag8(a.W3T + (size_t)col * 64 + 16 * k + lr);
    const float bj = a.w.b3[col];
    f4v dw[4];   // dW3(h = 16 th + lr + i, col)
#pragma unroll
    for (int th = 0; th < 4; ++th) dw[th] = f4v{0.f, 0.f, 0.f, 0.f};
    float db = 0.f;
    uint4 h0, h1, t0, t1;
    float xl = 0.f;   // this thread's of: 64 log-sum-exps of the tile's head, 64 weights, 64 bins' columns
    int xt = 0;
    auto load = [&](long long b) {
        h0 = ((const uint4*)(a.H2 + b * 4096))[tid];
        h1 = ((const uint4*)(a.H2 + b * 4096))[tid + 256];
        t0 = ((const uint4*)(a.H2T + b * 4096))[tid];
        t1 = ((const uint4*)(a.H2T + b * 4096))[tid + 256];
        const long long r = b * 64 + (tid & 63);
        if (tid < 64) xl = a.lse[2 * r + (jt > 0 ? 1 : 0)];
        else if (tid < 128) xl = a.sw[r];
        else if (tid < 192) xt = r < a.n ? (jt > 0 ? kMlpDir + a.tb[r] : a.td[r]) : -1;
    };
    auto put = [&](int p) {
        put_w3_tile(h0, h1, sH[p]);
        put_w3_tile(t0, t1, sHT[p]);
        if (tid < 64) slse[p][tid] = xl;
        else if (tid < 128) ssw[p][tid - 64] = xl;
        else if (tid < 192) shot[p][tid - 128] = xt;
    };
    if (b0 < b1) {
        load(b0);
        put(0);
    }
    for (long long b = b0; b < b1; ++b) {
        const int p = (int)(b - b0) & 1;
        load(b + 1 < b1 ? b + 1 : b);
        lds_sync();
        s4v dv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {   // 16 rows
            f4v acc = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 4; ++k) acc = DN_MFMA(frag8(sH[p] + (16 * q + lc) * PS + 16 * k + lr), wf[k], acc);
            const f4v lse = *(const f4v*)(slse[p] + 16 * q + lr), w = *(const f4v*)(ssw[p] + 16 * q + lr);
            const int4 hot = *(const int4*)(shot[p] + 16 * q + lr);
            const float d0 = mlp_dz(acc[0] + bj, w[0], lse[0], hot.x == col), d1 = mlp_dz(acc[1] + bj, w[1], lse[1], hot.y == col);
            const float d2 = mlp_dz(acc[2] + bj, w[2], lse[2], hot.z == col), d3 = mlp_dz(acc[3] + bj, w[3], lse[3], hot.w == col);
            db += used ? (d0 + d1) + (d2 + d3) : 0.f;
            dv[q] = used ? pack4(d0, d1, d2, d3) : s4v{0, 0, 0, 0};
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int th = 0; th < 4; ++th) dw[th] = DN_MFMA(frag8(sHT[p] + (16 * th + lc) * PS + 16 * q + lr), dv[q], dw[th]);
        put(p ^ 1);
    }
    float* part = a.part3 + (size_t)blockIdx.y * (64 + 1) * noutp;
#pragma unroll
    for (int th = 0; th < 4; ++th)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[(size_t)(16 * th + lr + i) * noutp + col] = dw[th][i];
    db += __shfl_xor(db, 16);
    db += __shfl_xor(db, 32);
    if (lane < 16) part[(size_t)64 * noutp + col] = db;
}

// grad: the parameters below W3 summed over the row blocks in order (64 per
// block here: a wave with 32 loads in flight), W3 and b3 over the splits; loss.
__global__ __launch_bounds__(256) void mlp_reduce(const float* part, const float* loss_part, int nblk, const float* part3,
                                                  int nsplit, int P, float* grad, float* loss)
{
    __shared__ float s[256];
    const int tid = threadIdx.x;
    constexpr int nsb = kMlpSmall / 64;
    if ((int)blockIdx.x < nsb) {
        if (tid < 64) {
            const float* q = part + blockIdx.x * 64 + tid;
            float v = 0.f;
            int b = 0;
            for (; b + 32 <= nblk; b += 32) {
                float x[32];
#pragma unroll
                for (int u = 0; u < 32; ++u) x[u] = q[(size_t)(b + u) * kMlpSmall];
#pragma unroll
                for (int u = 0; u < 32; ++u) v += x[u];
            }
            for (; b < nblk; ++b) v += q[(size_t)b * kMlpSmall];
            grad[blockIdx.x * 64 + tid] = v;
        }
        if (blockIdx.x == 0) {
            float l = 0.f;
            for (int i = tid; i < nblk; i += 256) l += loss_part[i];
            s[tid] = l;
            __syncthreads();
            for (int o = 128; o > 0; o >>= 1) {
                if (tid < o) s[tid] += s[tid + o];
                __syncthreads();
            }
            if (tid == 0) *loss = s[0];
        }
        return;
    }
    const int p = kMlpSmall + (blockIdx.x - nsb) * 256 + tid;
    if (p >= P) return;
    const size_t st = (size_t)(P - kMlpSmall);
    const float* q = part3 + (p - kMlpSmall);
    float v = 0.f;
    int k = 0;
    for (; k + 8 <= nsplit; k += 8) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = q[(size_t)(k + u) * st];
#pragma unroll
        for (int u = 0; u < 8; ++u) v += x[u];
    }
    for (; k < nsplit; ++k) v += q[(size_t)k * st];
    grad[p] = v;
}

// Adam on the FP32 master parameters; BF16 copies of the weight matrices.
__global__ void mlp_adam(float* theta, float* m, float* v, const float* grad, int P, MlpLayout L, float lr, float b1,
                         float b2, float eps, float c1, float c2, uint16_t* W1b, uint16_t* W2b, uint16_t* W3b)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const float g = grad[p];
    const float mm = b1 * m[p] + (1.f - b1) * g;
    const float vv = b2 * v[p] + (1.f - b2) * g * g;
    m[p] = mm;
    v[p] = vv;
    const float t = theta[p] - lr * (mm * c1) / (sqrtf(vv * c2) + eps);
    theta[p] = t;
    if (p >= L.oW1 && p < L.ob1) W1b[p - L.oW1] = f2bf(t);
    else if (p >= L.oW2 && p < L.ob2) W2b[p - L.oW2] = f2bf(t);
    else if (p >= L.oW3 && p < L.ob3) W3b[p - L.oW3] = f2bf(t);
}

// BF16 copies of the weight matrices of theta (after loading parameters).
__global__ void mlp_to_bf16(const float* theta, int P, MlpLayout L, uint16_t* W1b, uint16_t* W2b, uint16_t* W3b)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const float t = theta[p];
    if (p >= L.oW1 && p < L.ob1) W1b[p - L.oW1] = f2bf(t);
    else if (p >= L.oW2 && p < L.ob2) W2b[p - L.oW2] = f2bf(t);
    else if (p >= L.oW3 && p < L.ob3) W3b[p - L.oW3] = f2bf(t);
}

// Forward pass for n rows (64 per block): logits Z[n][noutp] (tests).
__global__ __launch_bounds__(256) void mlp_forward_rows(const float* X, long long n, MlpWeights w, float* Z)
{
    extern __shared__ float lds[];
    float* sX = lds;
    uint16_t* sH1b = (uint16_t*)(sX + 64 * kMlpIn);
    uint16_t* sH2b = sH1b + 4096;
    uint16_t* sW2b = sH2b + 4096;
    uint16_t* sW3b = sW2b + 4096;
    const long long r0 = (long long)blockIdx.x * 64;
    const int nrow = (int)((n - r0) < 64 ? (n - r0) : 64);
    for (int e = threadIdx.x; e < 64 * kMlpIn; e += blockDim.x) {
        const int s = e / kMlpIn;
        sX[e] = s < nrow ? X[(r0 + s) * kMlpIn + (e - s * kMlpIn)] : 0.f;
    }
    for (int e = threadIdx.x; e < 4096; e += blockDim.x) sW2b[e] = w.W2[e];
    __syncthreads();
    layer1(sX, w, nrow, sH1b);
    __syncthreads();
    {
        f4v acc[2][2];
        acc_zero(acc);
        gemm64(sH1b, 64, 1, sW2b, 64, 1, 64, acc);
        acc_each(acc, [&](int r, int c, float v) { sH2b[r * 64 + c] = f2bf(r < nrow ? tanhf(v + w.b2[c]) : 0.f); });
    }
    __syncthreads();
    for (int jt = 0; jt < w.noutp / 64; ++jt) {
        for (int e = threadIdx.x; e < 4096; e += blockDim.x) sW3b[e] = w.W3[(size_t)(e >> 6) * w.noutp + jt * 64 + (e & 63)];
        __syncthreads();
        f4v acc[2][2];
        acc_zero(acc);
        gemm64(sH2b, 64, 1, sW3b, 64, 1, 64, acc);
        acc_each(acc, [&](int r, int c, float v) {
            if (r < nrow) Z[(r0 + r) * w.noutp + jt * 64 + c] = v + w.b3[jt * 64 + c];
        });
        __syncthreads();
    }
}

// ------------------------------------------------------------ features ----
// Direction bin of descriptor words: 8 equal-area cos(theta) bins x 8 phi bins.
__device__ __forceinline__ int desc_dir_bin(uint32_t w0, uint32_t w1)
{
    return (int)(((w0 & 0xFFFFFFu) >> 21) * 8u + ((w1 & 0xFFFFFFu) >> 21));
}

// Training samples from the last plain run (records on, one batch): per ray
// its cell's features, direction bin, (band, g) bin and weight
// |x| / sqrt(steps + cost0), x = w D - winv G the ray's net contribution.  With
// cost0 < 0 the weight is |x|.  The |x|-weighted fit targets the
// zero-variance density p|x|; dividing by the square root of the ray's cost
// targets p|x|/sqrt(c), the density of least variance x cost.
__global__ void mlp_samples(FeatArgs f, const int4* slotinfo, long long slot0, int R, long long nrays, int nQ,
                            const uint32_t* w0, const uint32_t* w1, const float* wv, const float* winv,
                            const float* recD, const float* recG, const int* recS, float cost0, float* X, int* td,
                            int* tb, float* wt)
{
    for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < nrays; q += (long long)gridDim.x * blockDim.x) {
        const int4 si = slotinfo[slot0 + q / R];
        const int i = si.w & 1023, j = (si.w >> 10) & 1023, k = (si.w >> 20) & 1023;
        float x[kMlpIn];
        cell_features(f, i, j, k, x);
        for (int t = 0; t < kMlpIn; ++t) X[q * kMlpIn + t] = x[t];
        td[q] = desc_dir_bin(w0[q], w1[q]);
        tb[q] = desc_band(w0[q], w1[q]) * nQ + desc_g(w1[q]);
        const float xr = fabsf(wv[q] * recD[q] - winv[q] * recG[q]);
        wt[q] = cost0 < 0.f ? xr : xr * rsqrtf((float)recS[q] + cost0);
    }
}

// Features of the first n slots' cells (tests).
__global__ void mlp_features(FeatArgs f, const int4* slotinfo, long long n, float* X)
{
    for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < n; q += (long long)gridDim.x * blockDim.x) {
        const int4 si = slotinfo[q];
        float x[kMlpIn];
        cell_features(f, si.w & 1023, (si.w >> 10) & 1023, (si.w >> 20) & 1023, x);
        for (int t = 0; t < kMlpIn; ++t) X[q * kMlpIn + t] = x[t];
    }
}

// -------------------------------------------------- learned ray generation --
// mlp_proposal: one block per 64 consecutive slots, one pass over the output
// tiles.  The network's logits of the 64 cells (MFMA), e = exp(clamp(z)) and
// the running (unnormalised) sums per head written to U[slot][noutp]:
// columns [0, 64) the direction head, [64, 64 + nbin) the (band, g) head.
// The sampler normalises by the head's last entry and forms the defensive
// mixture on the fly, so no second pass over the logits is needed.
//
// A wave has 16 cells to itself from layer 2 on: their H2 fragments stay in
// registers, the logits come out transposed (four consecutive columns of a cell
// per lane), and the tile's exponentials, running sums and rows pass through
// its own rows of sZ, so the block meets once per 64 columns, for the W3 tile
// (two buffers).  The rows leave 4 x 256 bytes per store.  4.2e6 cells x 1664
// columns (28 GB): 10.2 -> 7.6 ms (three barriers per tile and 16-byte pieces
// 64 bytes apart before); three blocks per CU, four spill registers: 8.9 ms.
__global__ __launch_bounds__(256) void mlp_proposal(GenArgs a, float* U)
{
    // LDS (mlp_proposal_lds()): rows of kPropStride elements, so that MFMA
    // operand fragments (four consecutive BF16 of one row, one 8-byte read)
    // and the row scans are free of bank conflicts
    extern __shared__ __align__(16) float lds[];
    constexpr int PS = kPropStride;
    float* sX = lds;                                  // 64 x 6 features
    float* sZ = sX + 64 * kMlpIn;                     // 64 x PS: exp(z) of a column tile, then the running sums
    uint16_t* sW2T = (uint16_t*)sZ;                   //   (W2^T during layer 2)
    uint16_t* sW3T = (uint16_t*)(sZ + 64 * PS);       // 2 x 64 x PS: H1 and H2, then the W3^T tiles
    uint16_t *sH1b = sW3T, *sH2b = sW3T + 64 * PS;
    const int noutp = a.mlpw.noutp, nbin = a.mlpw.nbin, ntile = noutp / 64;
    const int tid = threadIdx.x, lane = tid & 63, wr = (tid >> 6) * 16;
    const int lc = lane & 15, lr = 4 * (lane >> 4);
    FeatArgs f = a.feat;
    f.T0 = a.T0 + (size_t)a.snap * a.tstride0;
    const int row = tid >> 2, part = tid & 3;         // 4 threads per row (of the wave), 16 columns each
    const long long ngroups = (a.nslots + 63) / 64;
    for (long long grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
        const long long s0 = grp * 64;
        const int ns = (int)((a.nslots - s0) < 64 ? (a.nslots - s0) : 64);
        __syncthreads();                              // (the last group's tiles are read)
        for (int e = tid; e < 64 * kMlpIn; e += blockDim.x) sX[e] = 0.f;
        // W2^T (64 rows of 64 BF16) into the padded rows of the sZ region
        for (int e = tid; e < 512; e += blockDim.x) {
            const uint4 r = ((const uint4*)a.mlpw.W2T)[e];
            uint2* d = (uint2*)(sW2T + (e >> 3) * PS + (e & 7) * 8);
            d[0] = make_uint2(r.x, r.y);
            d[1] = make_uint2(r.z, r.w);
        }
        __syncthreads();
        if (tid < ns) {
            const int4 si = a.slotinfo[a.slot0 + s0 + tid];
            cell_features(f, si.w & 1023, (si.w >> 10) & 1023, (si.w >> 20) & 1023, sX + tid * kMlpIn);
        }
        __syncthreads();
        layer1(sX, a.mlpw, ns, sH1b, PS);
        __syncthreads();
        {
            f4v acc[2][2];
            acc_zero(acc);
            gemm64(sH1b, PS, 1, sW2T, 1, PS, 64, acc);
            acc_each(acc, [&](int r, int c, float v) { sH2b[r * PS + c] = f2bf(r < ns ? tanhf(v + a.mlpw.b2[c]) : 0.f); });
        }
        __syncthreads();
        s4v ha[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) ha[k] = frag8(sH2b + (wr + lc) * PS + 16 * k + lr);
        float run = 0.f;                              // this row's running sum (held by all 4 lanes)
        // the W3 tile and this lane's b3 are loaded one tile ahead; the tile
        // loop's barrier waits for LDS traffic only
        uint4 t0, t1;
        float4 b3[4];
        auto bias = [&](int jt) {
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) b3[tj] = *(const float4*)(a.mlpw.b3 + jt * 64 + 16 * tj + lr);
        };
        load_w3_tile(a.mlpw.W3T, 0, t0, t1);
        bias(0);
        lds_sync();                                   // H1 and H2 are read: the tiles take their place
        put_w3_tile(t0, t1, sW3T);
        for (int jt = 0; jt < ntile; ++jt) {
            const uint16_t* sW = sW3T + (jt & 1) * 64 * PS;
            const int jn = min(jt + 1, ntile - 1);    // (the last tile again at the end)
            load_w3_tile(a.mlpw.W3T, jn, t0, t1);
            lds_sync();
            f4v acc[4];
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) acc[tj] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int tj = 0; tj < 4; ++tj)
                    acc[tj] = DN_MFMA(frag8(sW + (16 * tj + lc) * PS + 16 * k + lr), ha[k], acc[tj]);
            const int nc = kMlpDir + nbin - jt * 64 - lr;   // columns of a head from this lane's first on
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                const float bj[4] = {b3[tj].x, b3[tj].y, b3[tj].z, b3[tj].w};
                f4v e;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float z = fminf(fmaxf(acc[tj][i] + bj[i], -60.f), 60.f);
                    e[i] = 16 * tj + i < nc ? __expf(z) : 0.f;
                }
                *(f4v*)(sZ + (wr + lc) * PS + 16 * tj + lr) = e;
            }
            bias(jn);
            put_w3_tile(t0, t1, sW3T + ((jt + 1) & 1) * 64 * PS);
            if (jt == 1) run = 0.f;                   // the (band, g) head starts
            float* zr = sZ + row * PS + part * 16;    // (this wave's rows of sZ only)
            f4v loc[4];
            float sum = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const f4v z = *(const f4v*)(zr + 4 * c);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sum += z[i];
                    loc[c][i] = sum;
                }
            }
            float excl = sum;                          // scan of the 4 segment totals
            for (int o = 1; o < 4; o <<= 1) {
                const float t = __shfl_up(excl, o, 4);
                if (part >= o) excl += t;
            }
            const float total = __shfl(excl, 3, 4);
            excl -= sum;
            const float b0 = run + excl;
#pragma unroll
            for (int c = 0; c < 4; ++c) *(f4v*)(zr + 4 * c) = b0 + loc[c];
            run += total;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = wr + 4 * q + (lane >> 4), c = 4 * lc;
                const f4v v = *(const f4v*)(sZ + r * PS + c);
                if (r < ns) *(f4v*)(U + (s0 + r) * (size_t)noutp + jt * 64 + c) = v;
            }
        }
    }
}

// One learned ray: Philox (r, cell, snapshot, 1), the direction bin and the
// (band, g) bin from the defensive mixtures on the cell's row Ud (mix_search
// on each head), the direction uniform inside its bin, and p/q into the
// descriptor words of ray q.
__device__ __forceinline__ void learned_ray(const GenArgs& a, const float* Ud, const float* sPd, const float* sP,
                                            uint32_t r, uint32_t cell, long long q)
{
    const u32x4 x = philox4x32_10(u32x4{r, cell, (uint32_t)a.snap, 1u}, (uint32_t)a.seed, (uint32_t)(a.seed >> 32));
    float qd, qb;
    const int d = mix_search(Ud, sPd, kMlpDir, a.mix_eps, u01_open(x.x), &qd);
    const int bg = mix_search(Ud + kMlpDir, sP, a.mlpw.nbin, a.mix_eps, u01_open(x.y), &qb);
    const int band = bg / a.nQ, g = bg - band * a.nQ;
    // (a selected bin always has a positive step; the guard keeps a
    // degenerate row from producing inf * 0)
    const float ratio = (qb > 0.f && qd > 0.f) ? (a.p_bg[bg] / qb) * ((1.0f / kMlpDir) / qd) : 0.f;
    const uint32_t mt = ((uint32_t)(d >> 3) << 21) | (x.z >> 11);
    const uint32_t mp = ((uint32_t)(d & 7) << 21) | (x.w >> 11);
    uint32_t w0, w1;
    desc_pack(mt, mp, band, g, &w0, &w1);
    a.w0[q] = w0;
    a.w1[q] = w1;
    a.w[q] = ratio;
}

// raygen_learned: one thread per ray.  Each ray draws Philox (r, cell,
// snapshot, 1), its direction bin and (band, g) bin from the defensive
// mixtures by binary search on its cell's row of U (global memory: the R rays
// of a cell run in neighbouring lanes, so their first probes coincide and the
// rest hit the caches) and its direction uniform inside the bin.  The plain
// (band, g) CDF is in LDS.  The descriptor's w word carries p/q; the
// traversal multiplies it into the emission weight it computes from its LDS
// tables at ray start.
__global__ __launch_bounds__(256) void raygen_learned(GenArgs a, const float* U, const float* pcdf)
{
    extern __shared__ float lds[];
    const int noutp = a.mlpw.noutp, nbin = a.mlpw.nbin;
    float* sP = lds;
    for (int e = threadIdx.x; e < nbin; e += blockDim.x) sP[e] = pcdf[e];
    __shared__ float sPd[kMlpDir];
    for (int e = threadIdx.x; e < kMlpDir; e += blockDim.x) sPd[e] = (float)(e + 1) * (1.0f / kMlpDir);
    __syncthreads();
    const int R = a.rays_per_slot;
    const long long nr = a.nslots * (long long)R;
    for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < nr; q += (long long)gridDim.x * blockDim.x) {
        const long long sl = q / R;
        learned_ray(a, U + sl * (size_t)noutp, sPd, sP, (uint32_t)(q - sl * R), (uint32_t)a.slotinfo[a.slot0 + sl].y, q);
    }
}

// raygen_learned_lds: the same draws with the rows of G consecutive slots
// staged in LDS per block (G = 1..8 by the host: at 200 rays per cell and
// more the staging is shared by enough rays that the LDS probes' short
// latency pays for it).  Rays t of the group: slot t / R, ray t % R.
__global__ __launch_bounds__(256) void raygen_learned_lds(GenArgs a, const float* U, const float* pcdf, int G)
{
    extern __shared__ float lds[];
    const int noutp = a.mlpw.noutp, nbin = a.mlpw.nbin;
    float* sP = lds + G * noutp + 4;                  // (after the rows and one 16-byte pad slot)
    for (int e = threadIdx.x; e < nbin; e += blockDim.x) sP[e] = pcdf[e];
    __shared__ float sPd[kMlpDir];
    for (int e = threadIdx.x; e < kMlpDir; e += blockDim.x) sPd[e] = (float)(e + 1) * (1.0f / kMlpDir);
    __shared__ int s_cell[8];
    const int R = a.rays_per_slot;
    const long long ngroups = (a.nslots + G - 1) / G;
    const int npad = G * noutp / 4;                   // the pad slot (float4 index)
    for (long long grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
        const long long s0 = grp * G;
        const int ns = (int)((a.nslots - s0) < G ? (a.nslots - s0) : G);
        // the rows into LDS, eight 16-byte loads in flight per thread (no
        // branch between them: loads past the rows read the last element
        // again, their stores go to the pad slot, which nothing reads)
        const float4* src = (const float4*)(U + s0 * (size_t)noutp);
        float4* dst = (float4*)lds;
        const int nv = ns * noutp / 4;
        for (int e0 = (int)threadIdx.x; e0 < nv; e0 += 8 * (int)blockDim.x) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = src[min(e0 + u * (int)blockDim.x, nv - 1)];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int e = e0 + u * (int)blockDim.x;
                dst[e < nv ? e : npad] = v[u];
            }
        }
        if ((int)threadIdx.x < ns) s_cell[threadIdx.x] = a.slotinfo[a.slot0 + s0 + threadIdx.x].y;
        __syncthreads();
        for (int t = threadIdx.x; t < ns * R; t += blockDim.x) {
            const int sl = t / R, r = t - sl * R;
            learned_ray(a, lds + sl * noutp, sPd, sP, (uint32_t)r, (uint32_t)s_cell[sl], (s0 + sl) * (long long)R + r);
        }
        __syncthreads();
    }
}

}  // namespace dn
