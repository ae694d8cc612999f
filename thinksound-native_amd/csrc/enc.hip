// enc.hip — kernels of the text encoders (src/clip.cpp, src/t5.cpp): f32 GEMM over streamed f32 weights,
// LayerNorm with weight and bias, RMSNorm with weight, attention over one short context with the
// CLIP causal/EOT mask or the T5 bucketed relative bias and padding mask, quick GELU / GEGLU, and the
// token (+ position) embedding gather. GEMM operands are sums of three bf16 parts, which hold all 24 bits of
// an f32 value over f32's range of exponents (T5's activations leave the f16 range, and a row's values
// may lie any number of powers of two apart); everything else is f32.
//
// Per layer: norm -> QKV GEMM -> attention -> out GEMM -> norm -> FFN GEMM -> activation -> FFN GEMM.
// A GEMM leaves the raw sums of its K splits in the workspace; the kernel that reads them adds the
// splits in order with the bias (and the residual), so no GEMM has a reduce launch of its own, and
// writes its result as the next GEMM's operand (pack_parts4).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "dpp.h"

namespace tsn {

namespace {

typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef unsigned uintx4_t __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float floatx2_t __attribute__((ext_vector_type(2)));

// The three parts of N values: p[0] = bf16(v), p[1] = bf16(v - p[0]), p[2] = the rest, exact (8 + 8 + 8 bits).
// Two values a 32-bit word.
template <int N>
__device__ __forceinline__ void split_bf16(const float (&v)[N], unsigned (&p)[3][N / 2]) {
#pragma unroll
    for (int e = 0; e < N; e += 2) {
        floatx2_t r = {v[e], v[e + 1]};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2_t));
            p[c][e / 2] = u;
            r[0] -= __uint_as_float(u << 16);
            r[1] -= __uint_as_float(u & 0xFFFF0000u);
        }
    }
}

// A GEMM operand with M <= 16 mt rows, packed for enc_gemm_kernel: per 32-wide K step the three parts one
// after the other, each mt blocks of 16 rows x 32 columns (1 KB). A block is the 64 16-byte
// operands of one MFMA: row r (0..15), columns 8 kq .. + 7 (kq 0..3) at slot 4 r + (kq ^ (r / 2 % 4)).
// The slots of one row are 64 contiguous bytes (producers write one row), and the xor makes the reads of
// 8 lanes cover 128 contiguous bytes.
__device__ __forceinline__ int pack_slot(int r, int kq) { return 4 * r + (kq ^ ((r >> 1) & 3)); }
// columns k .. k + 3 (k % 4 == 0) of row m
__device__ __forceinline__ void pack_parts4(uint16_t *Ap, int mt, int m, int k, const float (&v)[4]) {
    unsigned p[3][2];
    split_bf16<4>(v, p);
    uint16_t *d = Ap + (((long long)(k >> 5) * 3 * mt + (m >> 4)) * 64 + pack_slot(m & 15, (k & 31) >> 3)) * 8 + (k & 4);
#pragma unroll
    for (int c = 0; c < 3; ++c) *(uint2 *)(d + c * mt * 512) = make_uint2(p[c][0], p[c][1]);
}

__device__ __forceinline__ float4 add4(float4 a, float4 b) {
    return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
// v[i] = the sum over the splits, in order, of the 4 columns at element off[i] of a GEMM's result. B splits
// are loaded at a time (past the last one, that one again, not added), so a reader waits for memory
// splits / B times, not once per split: these kernels are latency-bound.
template <int NV, int B>
__device__ __forceinline__ void parts_sum(const EncParts &p, const int (&off)[NV], float4 (&v)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int z = 0; z < p.splits; z += B) {
        float4 t[B][NV];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const float *s = p.ws + min(z + b, p.splits - 1) * p.stride;
#pragma unroll
            for (int i = 0; i < NV; ++i) t[b][i] = *(const float4 *)(s + off[i]);
        }
#pragma unroll
        for (int b = 0; b < B; ++b)
            if (z + b < p.splits) {
#pragma unroll
                for (int i = 0; i < NV; ++i) v[i] = add4(v[i], t[b][i]);
            }
    }
}

// Weights in the order the GEMM reads them: blocks of 64 rows (output columns) x 64 columns of K, 16 KB
// each, K innermost. Inside a block, each of 4 waves has 4 KB (32 rows, 32 columns) as its four 1 KB loads:
// rows 16 j .. + 15, lane: row lane % 16, columns 8 (lane / 16) + 4 q .. + 3. Row-major weights took 8% more
// time: rows of 4 or 8 KB put the 64 rows that a workgroup touches at once on a few memory channels.
__global__ __launch_bounds__(256) void enc_weight_pack_kernel(const float *__restrict__ src, float *__restrict__ dst, int K) {
    const int s = blockIdx.x, t = blockIdx.y, nkt = gridDim.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float *d = dst + (((long long)t * nkt + s) * 4 + wave) * 1024 + lane * 4;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = t * 64 + (wave & 1) * 32 + j * 16 + (lane & 15);
        const int k = s * 64 + (wave >> 1) * 32 + (lane >> 4) * 8;
#pragma unroll
        for (int q = 0; q < 2; ++q)
            *(float4 *)(d + (j * 2 + q) * 256) = k < K ? *(const float4 *)(src + (long long)row * K + k + 4 * q)
                                                       : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// ws[z][M][N] = sums over K split z of A[M][K] W[N][K]^T, A and W packed.
//
// The bound is the weight stream: each weight is read once up to 80 rows (one tile holds them all; twice up to 128), so the
// design keeps HBM loads in flight and everything else under them. Weights go straight from global
// memory to the registers of the lane that multiplies them (no LDS), three steps ahead, and are split
// there. Six v_mfma_f32_16x16x32_bf16 products (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi) replace eight
// f32 MFMAs of the same 32 columns of K at 3/8 of their matrix-core time; the dropped ones lie below 2^-24 of a
// product. The hi hi sums and the others have accumulators of their own, added at the end, so the
// main sum rounds once per 32 products instead of eight times: error against 64 bits of a T5 prompt
// 4.8e-7, 1.1e-6 on the f32 MFMA (CLIP 2.6e-7, 5.1e-7). 77 rows x 10240 x 2048: 28.8 us, 2.9 TB/s of weights.
// (Two f16 parts of rows scaled by a power of two took 23.1 us, but lost every bit of values 2^-39 of
// their row's largest, and splitting in the shadow of the MFMAs of the same wave took 31.4.)
//
// A step is 64 columns of K. 4 waves: wave w owns columns 32 (w & 1) .. + 31 of a 64-column tile and
// K half w >> 1 of every step, and the two halves' sums are added through LDS at the end, so each
// fragment of A read from LDS feeds two of W. A steps (6 KB per 16 rows) are shared by the waves through
// two LDS buffers, loaded two steps ahead (one with five row blocks, for registers: a step of fewer blocks is
// shorter than a load from L2; 2 T5 layers of 512, 8 rows: 83 us one step ahead, 71 two). Fetches past the split's end take its last step again, so
// every wait in the loop has a fixed count of younger loads to leave in flight.
//
// MTP: the operand's row blocks; with MTP > MT, blockIdx.z picks the MT of them that the workgroup takes.
template <int MT, int MTP>
__global__ __launch_bounds__(256, 2) void enc_gemm_kernel(const EncGemmArgs g) {
    constexpr int CH = 2 * 3 * MT * 64, NA = (CH + 255) / 256;   // 16-byte chunks of an A step, per thread
    constexpr int DA = MT < 5 ? 2 : 1;                           // steps that A is loaded ahead
    __shared__ __attribute__((aligned(16))) uintx4_t As[2][CH];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, kq = lane >> 4, wn = wave & 1, kh = wave >> 1;
    const int n0 = blockIdx.x * 64 + wn * 32, z = blockIdx.y, mb = MTP > MT ? blockIdx.z * MT : 0;
    const int nkt = (g.K + 63) >> 6;
    const int kt0 = z * g.kps, kt1 = min(nkt, kt0 + g.kps);
    const float *wb = g.W + ((long long)blockIdx.x * nkt * 4 + wave) * 1024;   // wave-uniform
    floatx4_t w[3][4];
    uintx4_t a[DA][NA];
    auto fetch_w = [&](int kt, floatx4_t (&d)[4]) {
        const floatx4_t *p = (const floatx4_t *)(wb + (long long)min(kt, kt1 - 1) * 4096);
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = p[(unsigned)(q * 64 + lane)];
    };
    auto full = [&](int i) { return CH % 256 == 0 || i < NA - 1 || wave < CH % 256 / 64; };   // wave-uniform
    auto fetch_a = [&](int kt, uintx4_t (&d)[NA]) {
        const uintx4_t *p = (const uintx4_t *)g.Ap + ((long long)min(kt, kt1 - 1) * 6 * MTP + mb) * 64;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int c = tid + 256 * i;
            if (full(i)) d[i] = p[(unsigned)(MTP > MT ? c / (64 * MT) * (64 * MTP) + c % (64 * MT) : c)];
        }
    };
    auto stash_a = [&](int b, const uintx4_t (&d)[NA]) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
            if (full(i)) As[b][tid + 256 * i] = d[i];
    };
    floatx4_t acc[2][MT], low[2][MT];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = low[j][i] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    const int slot = kh * 3 * MT * 64 + pack_slot(r16, kq);
    auto split_w = [&](const floatx4_t (&d)[4], bf16x8_t (&o)[2][3]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const floatx4_t x = d[2 * j], y = d[2 * j + 1];
            const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
            unsigned p[3][4];
            split_bf16<8>(v, p);
#pragma unroll
            for (int c = 0; c < 3; ++c) o[j][c] = __builtin_bit_cast(bf16x8_t, uintx4_t{p[c][0], p[c][1], p[c][2], p[c][3]});
        }
    };
    auto multiply = [&](int b, const bf16x8_t (&o)[2][3]) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {   // part c of A with parts 0 .. 2 - c of W
            bf16x8_t f[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) f[i] = __builtin_bit_cast(bf16x8_t, As[b][(c * MT + i) * 64 + slot]);
#pragma unroll
            for (int e = 0; e < 3 - c; ++e)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        floatx4_t &d = c + e == 0 ? acc[j][i] : low[j][i];
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o[j][e], f[i], d, 0, 0, 0);
                    }
        }
    };
    // Step kt issues A(kt + DA), then W(kt + 3) into the registers that W(kt) leaves: A(kt + 1) has to be in LDS
    // at the step's end, with the younger loads still in flight. LDS buffer (kt - kt0) & 1 holds A(kt); the
    // other one was last read in step kt - 1, before the barrier that ended it.
    fetch_a(kt0, a[0]);
    fetch_w(kt0, w[0]);
    fetch_w(kt0 + 1, w[1]);
    if constexpr (DA == 2) fetch_a(kt0 + 1, a[1]);
    else stash_a(0, a[0]);
    fetch_w(kt0 + 2, w[2]);
    if constexpr (DA == 2) stash_a(0, a[0]);
    __syncthreads();
    int kt = kt0;
    auto step = [&](int b, floatx4_t (&d)[4], uintx4_t (&in)[NA], const uintx4_t (&out)[NA]) {
        bf16x8_t o[2][3];
        fetch_a(kt + DA, in);
        split_w(d, o);
        fetch_w(kt + 3, d);
        multiply(b, o);
        stash_a(b ^ 1, out);
        __syncthreads();
        ++kt;
    };
    if constexpr (DA == 2) {
        while (kt + 6 <= kt1) {
#pragma unroll
            for (int u = 0; u < 6; ++u) step(u & 1, w[u % 3], a[u & 1], a[(u & 1) ^ 1]);
        }
#pragma unroll
        for (int u = 0; u < 5; ++u)   // the last zero to five steps
            if (kt < kt1) step(u & 1, w[u % 3], a[u & 1], a[(u & 1) ^ 1]);
    } else {
        int b = 0;
        while (kt + 3 <= kt1) {
#pragma unroll
            for (int u = 0; u < 3; ++u, b ^= 1) step(b, w[u], a[0], a[0]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u, b ^= 1)
            if (kt < kt1) step(b, w[u], a[0], a[0]);
    }
    // the weights are the first operand: a lane holds columns n0 + 16 j + 4 kq .. + 3 of row 16 i + r16;
    // 4 MT KB of the buffers' 12 MT
    floatx4_t *sum = (floatx4_t *)&As[0][0] + wn * 2 * MT * 64 + lane;
    if (kh > 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) sum[(j * MT + i) * 64] = acc[j][i] + low[j][i];
    }
    __syncthreads();
    if (kh > 0) return;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = 16 * (mb + i) + r16;
        if (m >= g.M) continue;
        float *y = g.ws + ((long long)z * g.M + m) * g.N + n0 + 4 * kq;
#pragma unroll
        for (int j = 0; j < 2; ++j) *(floatx4_t *)(y + 16 * j) = (acc[j][i] + low[j][i]) + sum[(j * MT + i) * 64];
    }
}

// One 256-thread workgroup per row: x += the previous GEMM's result (parts, if given; written back),
// then LayerNorm (w, b; mean, then variance of the centred row) or RMSNorm (w) of x as f32 rows (y)
// or as the next GEMM's operand (Ap). Sums are reduced per wave, then across the 4 waves in wave order.
// NJ: 1024-column groups of a row (H <= 1024 NJ, H % 4 == 0). ROWS: plain rows to plain rows, any number of them
// (tsn_ln_wb, tsn_rms_w), without the registers of the split sums.
template <bool LN, int NJ, bool ROWS>
__global__ __launch_bounds__(256) void enc_norm_kernel(const EncNormArgs a) {
    __shared__ float part[4];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, H = a.H;
    auto block_sum = [&](float v) {
        v = wave_sum(v);
        __syncthreads();   // part[] free from the previous reduction
        if (lane == 0) part[wave] = v;
        __syncthreads();
        return ((part[0] + part[1]) + part[2]) + part[3];
    };
    // the row in registers: columns 4*tid + 1024*j .. + 3; all loads ahead of the first barrier. Threads past the
    // row load its first columns: "in ? load : zero" became four loads of 4 bytes
    // (4096 x 1024: LN 14.3 us, now 6.5; RMS 10.8, now 5.6).
    float4 v[NJ], wv[NJ], bv[NJ];
    int off[NJ];   // of the GEMM's result, at most 128 rows; x and y may have any number (launch_enc_norm_rows)
    bool in[NJ];
    const float *xr = a.x + (long long)row * H;
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        in[j] = 4 * tid + 1024 * j < H;
        const int c = in[j] ? 4 * tid + 1024 * j : 0;
        off[j] = !ROWS && a.parts.ws ? row * H + c : 0;
        v[j] = *(const float4 *)(xr + c);
        wv[j] = *(const float4 *)(a.w + c);
        if (LN) bv[j] = *(const float4 *)(a.b + c);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        if (!in[j]) v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!ROWS && a.parts.ws) {
        float4 t[NJ], pb[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            pb[j] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (a.parts.bias) pb[j] = *(const float4 *)(a.parts.bias + (in[j] ? 4 * tid + 1024 * j : 0));
        }
        parts_sum<NJ, 8>(a.parts, off, t);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (in[j]) {
                v[j] = add4(v[j], add4(t[j], pb[j]));
                *(float4 *)(a.xout + off[j]) = v[j];
            }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        s += LN ? (v[j].x + v[j].y) + (v[j].z + v[j].w)
                : (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
    s = block_sum(s);
    float mean = 0.0f, inv;
    if (LN) {
        mean = s / (float)H;
        float q = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (in[j]) {
                const float d0 = v[j].x - mean, d1 = v[j].y - mean, d2 = v[j].z - mean, d3 = v[j].w - mean;
                q += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
            }
        q = block_sum(q);
        inv = 1.0f / sqrtf(q / (float)H + a.eps);
    } else {
        inv = 1.0f / sqrtf(s / (float)H + a.eps);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int c = 4 * tid + 1024 * j;
        if (!in[j]) continue;
        float4 o;
        if (LN) {
            o = make_float4((v[j].x - mean) * inv * wv[j].x + bv[j].x, (v[j].y - mean) * inv * wv[j].y + bv[j].y,
                            (v[j].z - mean) * inv * wv[j].z + bv[j].z, (v[j].w - mean) * inv * wv[j].w + bv[j].w);
        } else {
            o = make_float4(v[j].x * inv * wv[j].x, v[j].y * inv * wv[j].y, v[j].z * inv * wv[j].z, v[j].w * inv * wv[j].w);
        }
        if (!ROWS && a.Ap) {
            const float o4[4] = {o.x, o.y, o.z, o.w};
            pack_parts4(a.Ap, a.mt, row, c, o4);
        } else *(float4 *)(a.y + (long long)row * H + c) = o;
    }
}

constexpr int EA_Q = 16;      // queries per workgroup
constexpr int EA_SMAX = 128;  // longest context
constexpr int EA_HD = 64;
constexpr int EA_PP = EA_SMAX + 4;   // pitches (floats): the four k groups and sixteen rows or columns that
constexpr int EA_VP = EA_HD + 16;    // one MFMA operand read touches lie in distinct banks

// One workgroup per (16 queries, head), everything in f32 (v_mfma_f32_16x16x4_f32, f32 softmax). Wave w
// computes the scores of key block w (16 keys, MT of them at most) with k straight from the QKV GEMM's
// splits, then waves 0 to 3 the output columns 16 w .. + 15. The 64 products of a score run over
// d = 16 kq + i, so a lane's share of a k row is 64 contiguous bytes. The kernel is as long as its loads
// (77 keys, 4 splits: four waves with two key blocks and a q tile each 11.8 us, nine loads a thread and
// split instead of seventeen 9.2 us): q, k and v of up to 4 splits go out in one sequence.
template <int MT>
__global__ __launch_bounds__(64 * (MT < 4 ? 4 : MT), 1) void enc_attn_kernel(const EncAttnArgs a) {
    constexpr int NW = MT < 4 ? 4 : MT, NT = 64 * NW, VR = 256 * MT / NT;   // waves, threads, v rows of a thread
    constexpr int QP = EA_HD + 4;
    __shared__ __attribute__((aligned(16))) float Vs[16 * MT * EA_VP];
    __shared__ __attribute__((aligned(16))) float P[EA_Q * EA_PP];
    __shared__ __attribute__((aligned(16))) float Qs[EA_Q * QP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, kq = lane >> 4;
    // workgroups go to the 8 XCDs in turn: the query tiles of a head run on one XCD, whose L2 then serves
    // the head's k and v to all but the first of them
    const int S = a.S, H = a.nh * EA_HD, N = 3 * H, nkb = (S + 15) >> 4, idx = blockIdx.x >> 3;
    const int h = idx / nkb * 8 + (blockIdx.x & 7), q0 = idx % nkb * EA_Q;
    if (h >= a.nh) return;
    // q and v: 4 columns of row tid / 16 (of 16; + 4 NW i), k: columns 16 kq .. + 15 of row 16 wave + r16. Rows
    // past the context repeat its last one: masked, or never stored.
    constexpr int NV = 5 + VR;
    int off[NV];
    float4 x[NV];
    const int c4 = h * EA_HD + (tid & 15) * 4, ck = H + h * EA_HD + 16 * kq, cv = 2 * H + c4;
    off[0] = min(q0 + ((tid >> 4) & 15), S - 1) * N + c4;
#pragma unroll
    for (int i = 0; i < 4; ++i) off[1 + i] = min(16 * wave + r16, S - 1) * N + ck + 4 * i;
#pragma unroll
    for (int i = 0; i < VR; ++i) off[5 + i] = min((tid >> 4) + 4 * NW * i, S - 1) * N + cv;
    float4 bias[6];   // CLIP: q's, k's and v's columns
    if (a.qkv.bias) {
        bias[0] = *(const float4 *)(a.qkv.bias + c4);
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[1 + i] = *(const float4 *)(a.qkv.bias + ck + 4 * i);
        bias[5] = *(const float4 *)(a.qkv.bias + cv);
    }
    parts_sum<NV, 4>(a.qkv, off, x);
    if (a.qkv.bias) {
#pragma unroll
        for (int i = 0; i < NV; ++i) x[i] = add4(x[i], bias[i < 5 ? i : 5]);
    }
    if (tid < 256) *(float4 *)&Qs[(tid >> 4) * QP + (tid & 15) * 4] = x[0];
#pragma unroll
    for (int i = 0; i < VR; ++i) *(float4 *)&Vs[((tid >> 4) + 4 * NW * i) * EA_VP + (tid & 15) * 4] = x[5 + i];
    __syncthreads();
    const int q = q0 + r16;
    if (wave < nkb) {
        const int kb = wave;
        floatx4_t s = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 kv = x[1 + i], qv = *(const float4 *)&Qs[r16 * QP + 16 * kq + 4 * i];
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.x, qv.x, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.y, qv.y, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.z, qv.z, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.w, qv.w, s, 0, 0, 0);
        }
        // lane: keys 16 kb + 4 kq + r of query q
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 16 * kb + 4 * kq + r;
            s[r] *= a.scale;
            bool keep = k < S;
            if (a.mode == 1) {   // T5: padded keys masked, else the head's bias of the distance k - q
                keep = keep && (a.keys[k >> 5] >> (k & 31) & 1);
                if (keep && q < S) s[r] += a.rel[h * (2 * S - 1) + k - q + S - 1];
            } else {             // CLIP: causal, and nothing past the end-of-text token
                keep = keep && k <= q && k <= a.eot;
            }
            if (!keep) s[r] = -INFINITY;
        }
        *(floatx4_t *)&P[r16 * EA_PP + 16 * kb + 4 * kq] = s;
    }
    __syncthreads();
    // softmax: wave w takes queries w, w + NW, ..., one lane per key and 64 keys at a time
    for (int r = wave; r < EA_Q; r += NW) {
        float *pr = P + r * EA_PP;
        const int n = nkb * 16;
        const float s0 = lane < n ? pr[lane] : -INFINITY, s1 = lane + 64 < n ? pr[lane + 64] : -INFINITY;
        const float mx = wave_max(fmaxf(s0, s1));
        const float e0 = expf(s0 - mx), e1 = expf(s1 - mx);
        const float inv = 1.0f / wave_sum(e0 + e1);
        if (lane < n) pr[lane] = e0 * inv;
        if (lane + 64 < n) pr[lane + 64] = e1 * inv;
    }
    __syncthreads();
    if (wave >= 4) return;
    // V^T is the first operand: a lane holds columns 16 wave + 4 kq .. + 3 of query q
    floatx4_t o[2] = {floatx4_t{0.f, 0.f, 0.f, 0.f}, floatx4_t{0.f, 0.f, 0.f, 0.f}};
    for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * kb + 4 * i + kq;
            o[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(Vs[k * EA_VP + 16 * wave + r16], P[r16 * EA_PP + k],
                                                            o[i & 1], 0, 0, 0);
        }
    if (q >= S) return;
    const floatx4_t y = o[0] + o[1];
    const float y4[4] = {y[0], y[1], y[2], y[3]};
    pack_parts4(a.Ap, a.mt, q, h * EA_HD + 16 * wave + 4 * kq, y4);
}

// The FFN activation of a GEMM's result as the next GEMM's operand, four columns a thread: quick GELU of
// column c (shaders/ops_conv.metal:25-29), or gelu_tanh(column c) * column F + c (GEGLU; tanh form, argument
// clamped to +-10: shaders/ops_conv.metal:15-24).
template <bool GEGLU>
__global__ __launch_bounds__(256) void enc_act_kernel(EncParts p, uint16_t *Ap, int mt, int F) {
    constexpr int NV = GEGLU ? 2 : 1;
    const int m = blockIdx.y, c = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (c >= F) return;
    p.ws += (long long)m * p.N;
    int off[NV];
    float4 u[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) off[i] = i * F + c;
    parts_sum<NV, 4>(p, off, u);
    if (p.bias) {
#pragma unroll
        for (int i = 0; i < NV; ++i) u[i] = add4(u[i], *(const float4 *)(p.bias + i * F + c));
    }
    const float uv[4] = {u[0].x, u[0].y, u[0].z, u[0].w};
    float y[4];
    if constexpr (GEGLU) {
        const float gv[4] = {u[1].x, u[1].y, u[1].z, u[1].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = uv[e], t = 0.7978845608f * (v + 0.044715f * v * v * v);
            y[e] = 0.5f * v * (1.0f + tanhf(fminf(fmaxf(t, -10.0f), 10.0f))) * gv[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = uv[e] / (1.0f + expf(-1.702f * uv[e]));
    }
    pack_parts4(Ap, mt, m, c, y);
}

// x[s][c] = tok[ids[s]][c] (+ pos[s][c]), one workgroup per row; the ids are kernel arguments, so the
// call needs no copy to the device and no wait
__global__ __launch_bounds__(256) void embed_rows_kernel(const EncIds ids, const float *__restrict__ tok,
                                                         const float *__restrict__ pos, float *__restrict__ x, int H) {
    const int s = blockIdx.x;
    const float *t = tok + (long long)ids.id[s] * H;
    for (int c = threadIdx.x * 4; c < H; c += 1024) {
        float4 v = *(const float4 *)(t + c);
        if (pos) v = add4(v, *(const float4 *)(pos + (long long)s * H + c));
        *(float4 *)(x + (long long)s * H + c) = v;
    }
}

bool aligned16(const void *p) { return (((uintptr_t)p) & 15) == 0; }

} // namespace

// 2 T5 layers 2048 wide: 64 rows 202 us with five row blocks, 197 with four (512 wide 94 and 91)
int enc_row_blocks(int M) { return M <= 32 ? 2 : M <= 64 ? 4 : M <= 80 ? 5 : 8; }
size_t enc_operand_bytes(int M, int K) {   // whole 64-column steps
    return (size_t)3 * enc_row_blocks(M) * 16 * ((K + 63) / 64 * 64) * sizeof(uint16_t);
}

size_t enc_weight_floats(int N, int K) { return (size_t)N * ((K + 63) / 64 * 64); }

int launch_enc_weight_pack(const float *src, float *dst, int N, int K, hipStream_t st) {
    TSN_REQUIRE(src && dst && N > 0 && K > 0 && N % 64 == 0 && K % 32 == 0 && aligned16(src) && aligned16(dst),
                "enc_weight_pack: 16-byte aligned weights, N a multiple of 64, K of 32");
    // blocks of N in groups that the grid's second dimension takes
    const int nkt = (K + 63) / 64;
    for (int t0 = 0; t0 < N / 64; t0 += 65535) {
        const int n = std::min(65535, N / 64 - t0);
        TSN_LAUNCH(enc_weight_pack_kernel, dim3(nkt, n), dim3(256), 0, st, src + (size_t)t0 * 64 * K,
                   dst + (size_t)t0 * nkt * 4096, K);
    }
    TSN_HIP_CHECK(hipGetLastError());
    return TSN_OK;
}

int launch_enc_gemm(EncGemmArgs &g, hipStream_t st) {
    TSN_REQUIRE(g.Ap && g.W && g.ws && g.M > 0 && g.M <= 128 && g.N > 0 && g.K > 0,
                "enc_gemm: null operand, or rows outside 1..128");
    TSN_REQUIRE(g.N % 64 == 0 && g.K % 32 == 0, "enc_gemm: N a multiple of 64, K of 32");
    TSN_REQUIRE(aligned16(g.Ap) && aligned16(g.W) && aligned16(g.ws), "enc_gemm: 16-byte aligned operands");
    const int mt = enc_row_blocks(g.M);
    TSN_REQUIRE((size_t)g.M * g.N * sizeof(float) <= g.ws_bytes, "enc_gemm: workspace");
    // at most two workgroups per CU, of at least four steps each
    const int tiles = g.N / 64, steps = (g.K + 63) / 64;
    const int fit = (int)std::min<size_t>(std::max(1, steps / 4), g.ws_bytes / ((size_t)g.M * g.N * sizeof(float)));
    const int want = std::max(1, std::min(std::min(fit, g.most), 512 / tiles));
    g.kps = (steps + want - 1) / want;
    g.splits = (steps + g.kps - 1) / g.kps;
    const dim3 grid(tiles, g.splits, mt == 8 ? 2 : 1), block(256);   // more than 80 rows: two halves
    if (mt == 2) TSN_LAUNCH((enc_gemm_kernel<2, 2>), grid, block, 0, st, g);
    else if (mt == 4) TSN_LAUNCH((enc_gemm_kernel<4, 4>), grid, block, 0, st, g);
    else if (mt == 5) TSN_LAUNCH((enc_gemm_kernel<5, 5>), grid, block, 0, st, g);
    else TSN_LAUNCH((enc_gemm_kernel<4, 8>), grid, block, 0, st, g);
    TSN_HIP_CHECK(hipGetLastError());
    return TSN_OK;
}

int launch_enc_norm(const EncNormArgs &a, bool ln, hipStream_t st) {
    TSN_REQUIRE(a.x && a.w && (a.y || a.Ap) && a.rows > 0 && a.H > 0 && (!ln || a.b), "enc_norm: arguments");
    TSN_REQUIRE(!a.parts.ws || (a.xout && a.rows <= 128 && a.parts.splits > 0 && a.parts.N == a.H), "enc_norm: partial sums");
    TSN_REQUIRE(!a.Ap || (a.rows <= 128 && a.H % 32 == 0), "enc_norm: packed rows");
    TSN_REQUIRE(a.H % 4 == 0 && a.H <= 2048 && aligned16(a.x) && aligned16(a.y) && aligned16(a.w) && aligned16(a.b),
                "enc_norm: rows of at most 2048 floats, a multiple of 4, 16-byte aligned");
    const dim3 grid(a.rows), block(256);
    if (!a.parts.ws && !a.Ap) {
        if (ln && a.H <= 1024) TSN_LAUNCH((enc_norm_kernel<true, 1, true>), grid, block, 0, st, a);
        else if (ln) TSN_LAUNCH((enc_norm_kernel<true, 2, true>), grid, block, 0, st, a);
        else if (a.H <= 1024) TSN_LAUNCH((enc_norm_kernel<false, 1, true>), grid, block, 0, st, a);
        else TSN_LAUNCH((enc_norm_kernel<false, 2, true>), grid, block, 0, st, a);
    } else if (ln && a.H <= 1024) TSN_LAUNCH((enc_norm_kernel<true, 1, false>), grid, block, 0, st, a);
    else if (ln) TSN_LAUNCH((enc_norm_kernel<true, 2, false>), grid, block, 0, st, a);
    else if (a.H <= 1024) TSN_LAUNCH((enc_norm_kernel<false, 1, false>), grid, block, 0, st, a);
    else TSN_LAUNCH((enc_norm_kernel<false, 2, false>), grid, block, 0, st, a);
    TSN_HIP_CHECK(hipGetLastError());
    return TSN_OK;
}

int launch_enc_norm_rows(const float *x, float *y, const float *w, const float *b, int rows, int H, float eps, bool ln,
                         hipStream_t st) {
    TSN_REQUIRE(y, "enc_norm: arguments");
    EncNormArgs a{};
    a.x = x; a.y = y; a.w = w; a.b = b; a.rows = rows; a.H = H; a.eps = eps;
    return launch_enc_norm(a, ln, st);
}

int launch_enc_attention(const EncAttnArgs &a, hipStream_t st) {
    TSN_REQUIRE(a.qkv.ws && a.Ap && a.S > 0 && a.S <= EA_SMAX && a.nh > 0 && a.qkv.N == 3 * EA_HD * a.nh,
                "enc_attention: context 1..128, rows of q, k and v with heads of 64");
    TSN_REQUIRE((a.mode == 1 && a.rel) || a.mode == 2, "enc_attention: mode and tables");
    const dim3 grid((a.nh + 7) / 8 * 8 * ((a.S + EA_Q - 1) / EA_Q));
    const int mt = enc_row_blocks(a.S);
    if (mt == 2) TSN_LAUNCH(enc_attn_kernel<2>, grid, dim3(256), 0, st, a);
    else if (mt == 4) TSN_LAUNCH(enc_attn_kernel<4>, grid, dim3(256), 0, st, a);
    else if (mt == 5) TSN_LAUNCH(enc_attn_kernel<5>, grid, dim3(320), 0, st, a);
    else TSN_LAUNCH(enc_attn_kernel<8>, grid, dim3(512), 0, st, a);
    TSN_HIP_CHECK(hipGetLastError());
    return TSN_OK;
}

int launch_enc_act(const EncParts &p, bool geglu, uint16_t *Ap, int rows, int F, hipStream_t st) {
    TSN_REQUIRE(p.ws && Ap && rows > 0 && rows <= 128 && F > 0 && F % 32 == 0 && p.N == (geglu ? 2 * F : F),
                "enc_act: arguments");
    const dim3 grid((F + 1023) / 1024, rows), block(256);
    if (geglu) TSN_LAUNCH(enc_act_kernel<true>, grid, block, 0, st, p, Ap, enc_row_blocks(rows), F);
    else TSN_LAUNCH(enc_act_kernel<false>, grid, block, 0, st, p, Ap, enc_row_blocks(rows), F);
    TSN_HIP_CHECK(hipGetLastError());
    return TSN_OK;
}

int launch_embed_rows(const EncIds &ids, const float *tok, const float *pos, float *x, int S, int H, hipStream_t st) {
    TSN_REQUIRE(tok && x && S > 0 && S <= EA_SMAX && H > 0 && H % 4 == 0, "embed: arguments");
    TSN_LAUNCH(embed_rows_kernel, dim3(S), dim3(256), 0, st, ids, tok, pos, x, H);
    TSN_HIP_CHECK(hipGetLastError());
    return TSN_OK;
}

} // namespace tsn
