// q8_ops.hip -- the reference geometry's quantised ops on gfx950:
//   * GGML_OP_M4_WKB with a Q8_0 W_kb (patches/ggml-m4/m4-wkb.cu:14-86),
//   * GGML_OP_M4_PHASE phase 1, wv_b (m4-phase.cu:44-89, 209-224),
//   * GGML_OP_M4_PHASE phase 0, KV-write: wkv_a gemv, RMS norm, YaRN rope and the in-place f16
//     (or Q8_0) scatter into the cache (m4-phase.cu:91-200, 226-273).
// Numerics are the reference kernels' (the GPU MMVQ form, not ggml-cpu's): the f32 activation is
// quantised per 32-value block (d = amax / 127, an f16 scale, int8 quants by roundf(x / d) in
// WKB and roundf(x * (1 / d)) in the PHASE ops), block dots are exact int32 sums (v_dot4_i32_i8),
// and the f32 accumulation keeps the reference's order -- per row, or per lane and then the
// 32-lane xor butterfly of warp_reduce_sum -- so the integer paths match the CPU restatement bit
// for bit.  All three are small latency-bound launches (0.5 MiB, 1 MiB and 1.4 MiB of weights).
#include "mla_common.h"
#include "mla_kernels.h"

namespace mla {

namespace {

__device__ __forceinline__ float f16_bits(uint32_t bits) { return (float)__builtin_bit_cast(half_t, (uint16_t)bits); }
__device__ __forceinline__ float round_to_f16(float x) { return (float)(half_t)x; }

// The 4 bytes of a row at byte offset B, from the row's dwords D (B folds to a constant once the
// caller's loops are unrolled; rows are 4-byte aligned, Q8_0 blocks only 2-byte aligned).
__device__ __forceinline__ uint32_t bytes4(const uint32_t * D, int B) {
    const int i = B >> 2, r = B & 3;
    return r == 0 ? D[i] : __builtin_amdgcn_alignbyte(D[i + 1], D[i], r);
}

// Block quantisation with one value per lane of a 32-lane half-wavefront (the xor offsets stay
// inside the half): returns the int8 quant, d16 = the block's f16 scale as f32.
template <bool DIV>
__device__ __forceinline__ int quant_lane(float x, float & d16) {
    const float amax = half_max(fabsf(x));
    const float d = amax / 127.0f;
    d16 = round_to_f16(d);
    if constexpr (DIV) return amax == 0.0f ? 0 : (int)roundf(x / d);
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    return (int)roundf(x * id);
}

// The 32-lane butterfly of warp_reduce_sum (xor 16, 8, 4, 2, 1) inside a half-wavefront: the
// same additions in the same order (mla_common.h).
__device__ __forceinline__ float half_wave_sum(float v) { return half_sum(v); }

// ---- WKB, Q8_0 W_kb: one workgroup per (head, token); a thread per output row ----
// The head's d_n activations are quantised once into LDS (4 int8 per word); each row's blocks
// come in as dwords (17 per 2 blocks), the qs realigned with v_alignbyte, dotted with
// v_dot4_i32_i8, and acc = fma(wd * d16, sum, acc) over the blocks in order (m4-wkb.cu:30-52).
template <int NB>
__global__ __launch_bounds__(256) void wkb_q8_kernel(WkbArgs a) {
    static_assert(NB % 2 == 0, "rows of an even number of blocks are 4-byte aligned");
    constexpr int RW = NB * 17 / 2;      // dwords per row
    __shared__ uint32_t xq[NB * 8];
    __shared__ float xd[NB];
    const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x;
    if (tid < NB * 32) {                 // whole wavefronts: NB * 32 is a multiple of 64
        const float x = reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.q) + (size_t)t * a.q_nb2 +
                                                        (size_t)h * a.q_nb1)[tid];
        float d16;
        const int q = quant_lane<true>(x, d16);
        reinterpret_cast<int8_t *>(xq)[tid] = (int8_t)q;
        if ((tid & 31) == 0) xd[tid >> 5] = d16;
    }
    __syncthreads();
    float * drow = reinterpret_cast<float *>(reinterpret_cast<char *>(a.dst) + (size_t)t * a.d_nb2 + (size_t)h * a.d_nb1);
    for (int r = tid; r < a.d_v; r += 256) {
        const uint32_t * row = reinterpret_cast<const uint32_t *>(a.wq + ((size_t)h * a.d_v + r) * (NB * 34));
        uint32_t D[RW];
#pragma unroll
        for (int i = 0; i < RW; ++i) D[i] = row[i];
        float acc = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int o = 34 * b;
            const float wd = f16_bits((D[o >> 2] >> (8 * (o & 3))) & 0xffffu);
            int s = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) s = __builtin_amdgcn_sdot4((int)bytes4(D, o + 2 + 4 * j), (int)xq[8 * b + j], s, false);
            acc = fmaf(wd * xd[b], (float)s, acc);
        }
        drow[r] = acc;
    }
}

// ---- PHASE 1, wv_b: 8 outputs per workgroup (one per 32-lane half), grid (d_out / 8, H, nt) ----
// Lane k of an output's half holds element k of every block: p_k = sum_b fma(wd_b * xd_b,
// q_w[b][k] * q_x[b][k], .), then the butterfly (m4-phase.cu:52-88).
template <int NB>
__global__ __launch_bounds__(256) void wvb_q8_kernel(WvbArgs a) {
    __shared__ int8_t xq[NB * 32];
    __shared__ float xd[NB];
    const int h = blockIdx.y, t = blockIdx.z, tid = threadIdx.x;
    const float * xh = reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.x) + (size_t)t * a.x_nb1 +
                                                       (size_t)h * a.x_nb2);
    static_assert((NB * 32) % 256 == 0, "whole rounds of the workgroup");
#pragma unroll
    for (int i0 = 0; i0 < NB * 32; i0 += 256) {
        const int i = i0 + tid;
        float d16;
        const int q = quant_lane<false>(xh[i], d16);
        xq[i] = (int8_t)q;
        if ((i & 31) == 0) xd[i >> 5] = d16;
    }
    __syncthreads();
    const int o = blockIdx.x * 8 + (tid >> 5);
    const int k = tid & 31;
    if (o >= a.d_out) return;                // whole halves leave together
    const uint8_t * row = a.w + ((size_t)h * a.d_out + o) * (NB * 34);
    float acc = 0.0f;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const float wd = f16_bits(*reinterpret_cast<const uint16_t *>(row + 34 * b));
        const int q = (int)reinterpret_cast<const int8_t *>(row + 34 * b + 2)[k];
        acc = fmaf(wd * xd[b], (float)(q * (int)xq[32 * b + k]), acc);
    }
    acc = half_wave_sum(acc);
    if (k == 0)
        reinterpret_cast<float *>(reinterpret_cast<char *>(a.dst) + (size_t)t * a.d_nb1 + (size_t)h * a.d_nb2)[o] = acc;
}

// ---- several tokens (chunked prefill): wv_b and WKB as tiled products ----
// The per-token kernels above re-read the head's weights and re-quantise its activations for every
// few outputs of every token.  Here a workgroup takes 32 tokens of one head and quantises them once,
// into LDS.  Measured on the MI355X, 32 heads, per-token -> tiled kernel (us): wv_b 256 -> 128: 16
// tokens 7.9 -> 9.9, 24 10.9 -> 10.2, 64 24.5 -> 10.5, 500 212 -> 20.4; 512 -> 128: 16 14.0 -> 18.7,
// 24 19.8 -> 19.1, 64 48.8 -> 19.6.  WKB 64 -> 256: 32 tokens 3.0 -> 3.8, 64 4.4 -> 4.0, 500 22.3 ->
// 7.6; 128 -> 512: 16 4.4 -> 4.1, 64 16.0 -> 5.1, 500 111 -> 14.0.  The per-token kernels' time goes
// with their workgroups (or rows), the tiled ones' has a floor of one tile's latency, so the lines lie
// at a number of workgroups (wv_b: 24 tokens x 32 heads x 16) and at a number of rows times their
// length (WKB: 56 tokens x 32 heads x 256 rows x 64), and no tile is mostly empty below 8 tokens.
constexpr int Q8_GEMM_MIN_TOKENS = 8;
inline bool wvb_tiled(const WvbArgs & a) {
    return a.nt >= Q8_GEMM_MIN_TOKENS && (int64_t)a.nt * a.n_head * ((a.d_out + 7) / 8) >= 24 * 32 * 16 &&
           a.d_out <= 128 * 65535;          // its grid's y
}
inline bool wkb_q8_tiled(const WkbArgs & a) {
    return a.nt >= Q8_GEMM_MIN_TOKENS && (int64_t)a.nt * a.n_head * ((a.d_v + 255) / 256) * a.d_n >= 56 * 32 * 64;
}
constexpr int GT = 32;                   // tokens per workgroup
constexpr uint32_t Q_PAD = 16;           // LDS row padding: rows start on distinct banks

struct __attribute__((packed, aligned(4))) U4u { uint32_t v[4]; };       // as F4u

// Half a Q8 block of token r = lane & 31 (values 16 (lane >> 5) .. +15 of the block at x): its int8
// quants as 4 dwords and the block's scale, with quant_lane's arithmetic (the two halves of a block
// meet by v_permlane32_swap).
template <bool DIV>
__device__ __forceinline__ u32x4 quant_half_block(const F4u (&x)[4], float & d16) {
    float amax = fabsf(x[0].v[0]);
#pragma unroll
    for (int i = 1; i < 16; ++i) amax = fmaxf(amax, fabsf(x[i >> 2].v[i & 3]));
    float lo, hi;
    halves_pair(amax, lo, hi);
    amax = fmaxf(lo, hi);
    const float d = amax / 127.0f;
    d16 = round_to_f16(d);
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t wv = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = x[i].v[e];
            int q;
            if constexpr (DIV) q = amax == 0.0f ? 0 : (int)roundf(v / d);
            else q = (int)roundf(v * id);
            wv |= ((uint32_t)(uint8_t)(int8_t)q) << (8 * e);
        }
        r[i] = wv;
    }
    return r;
}

// The 16 int8 of half kh of block b of a Q8_0 row (4-byte aligned, an even number of blocks): the
// qs start 2 bytes past a dword in even blocks (a fifth dword, still inside the row, is read) and
// on one in odd blocks.
__device__ __forceinline__ u32x4 q8_half_block(const uint8_t * row, int b, int kh) {
    const uint8_t * p = row + 34 * b + 16 * kh;
    if (b & 1) {
        const U4u u = *reinterpret_cast<const U4u *>(p + 2);
        return u32x4{u.v[0], u.v[1], u.v[2], u.v[3]};
    }
    const U4u u = *reinterpret_cast<const U4u *>(p);
    const uint32_t e = *reinterpret_cast<const uint32_t *>(p + 16);
    return u32x4{__builtin_amdgcn_alignbyte(u.v[1], u.v[0], 2), __builtin_amdgcn_alignbyte(u.v[2], u.v[1], 2),
                 __builtin_amdgcn_alignbyte(u.v[3], u.v[2], 2), __builtin_amdgcn_alignbyte(e, u.v[3], 2)};
}
__device__ __forceinline__ float q8_value(const u32x4 & q, int j, float d) {
    return (float)(int)(int8_t)(uint8_t)(q[j >> 2] >> (8 * (j & 3))) * d;
}

// Quantise GT tokens of head h (rows of NB blocks at x + t x_nbt): the workgroup's waves take blocks
// w, w + 4, ...; quants to xq[token][NB * 32 + Q_PAD], scales to xd[block][token].
template <int NB, bool DIV>
__device__ __forceinline__ void quant_tokens(const char * x, int64_t x_nbt, int t0, int nt, char * xq, float (*xd)[GT]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 31, kh = lane >> 5;
    const float * row = reinterpret_cast<const float *>(x + (size_t)min(t0 + r, nt - 1) * x_nbt) + 16 * kh;
    constexpr int BPW = (NB + 3) / 4;
    F4u v[BPW][4];
#pragma unroll
    for (int i = 0; i < BPW; ++i)
        if (w + 4 * i < NB) {
#pragma unroll
            for (int k = 0; k < 4; ++k) v[i][k] = *reinterpret_cast<const F4u *>(row + 32 * (w + 4 * i) + 4 * k);
        }
#pragma unroll
    for (int i = 0; i < BPW; ++i) {
        const int b = w + 4 * i;
        if (b < NB) {
            float d16;
            const u32x4 q = quant_half_block<DIV>(v[i], d16);
            *reinterpret_cast<u32x4 *>(xq + r * (NB * 32 + Q_PAD) + 32 * b + 16 * kh) = q;
            if (kh == 0) xd[b][r] = d16;
        }
    }
}

// wv_b over 32 tokens x 128 outputs of one head: wave w takes outputs 32 w .. +31.
// The per-token kernel's result is, per element position k of a block, a chain over the blocks of
// fma(wd_b xd_b, qw qx, .), then the butterfly over k.  wd_b xd_b (two f16 scales), qw wd_b and
// qx xd_b are exact in f32, so each link is also fma(qw wd_b, qx xd_b, .): an outer product over
// (token, output) per (k, b), which v_mfma_f32_32x32x1_2b_f32 (K = 1: one fused multiply-add per
// element) computes with the same single rounding.  Its two blocks take positions j and j + 16, whose
// sums are the butterfly's first step; the other steps are additions of accumulators in the
// butterfly's order (16, 8, 4, 2, 1), so the result is the per-token kernel's bit for bit.
// Bound: its MFMAs, 16 NB of 64 cycles per wave (NB = 8, 500 tokens x 32 heads: 2,048 waves, two per
// SIMD, 6.8 us); 20.4 us there against 212 us for the per-token kernel.
template <int NB>
__global__ __launch_bounds__(256, NB <= 8 ? 2 : 1) void wvb_q8_gemm_kernel(WvbArgs a) {
    static_assert(NB % 2 == 0 && NB >= 4, "rows of an even number of blocks are 4-byte aligned");
    __shared__ __attribute__((aligned(16))) char xq[GT * (NB * 32 + Q_PAD)];
    __shared__ float xd[NB][GT];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 31, kh = lane >> 5;
    const int t0 = blockIdx.x * GT, o0 = blockIdx.y * 128 + 32 * w, h = blockIdx.z;
    // B operand: column o0 + r, element positions 16 kh + j of every block
    const uint8_t * wrow = a.w + ((size_t)h * a.d_out + min(o0 + r, a.d_out - 1)) * (NB * 34);
    u32x4 qw[NB];
    float wd[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        qw[b] = q8_half_block(wrow, b, kh);
        wd[b] = f16_bits(*reinterpret_cast<const uint16_t *>(wrow + 34 * b));
    }
    quant_tokens<NB, false>(reinterpret_cast<const char *>(a.x) + (size_t)h * a.x_nb2, a.x_nb1, t0, a.nt, xq, xd);
    __syncthreads();
    if (o0 >= a.d_out) return;               // whole waves leave together
    // A operand: token t0 + r, the same element positions
    u32x4 qx[NB];
    float xs[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        qx[b] = *reinterpret_cast<const u32x4 *>(xq + r * (NB * 32 + Q_PAD) + 32 * b + 16 * kh);
        xs[b] = xd[b][r];
    }
    typedef float f32x32 __attribute__((ext_vector_type(32)));
    // positions j, j + 16, j + 8 and j + 24 of the block: two chains, then the first two butterfly steps
    auto s8 = [&](int j) __attribute__((always_inline)) {
        f32x32 c0, c1;
#pragma unroll
        for (int i = 0; i < 32; ++i) { c0[i] = 0.0f; c1[i] = 0.0f; }
        // the operands of block b + 1 are converted under the MFMAs of block b; the scheduling
        // barriers keep the compiler from converting every block first (and spilling)
        float xa = q8_value(qx[0], j, xs[0]), xb = q8_value(qx[0], j + 8, xs[0]);
        float ya = q8_value(qw[0], j, wd[0]), yb = q8_value(qw[0], j + 8, wd[0]);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            c0 = __builtin_amdgcn_mfma_f32_32x32x1f32(xa, ya, c0, 0, 0, 0);
            c1 = __builtin_amdgcn_mfma_f32_32x32x1f32(xb, yb, c1, 0, 0, 0);
            if (b + 1 < NB) {
                xa = q8_value(qx[b + 1], j, xs[b + 1]);
                xb = q8_value(qx[b + 1], j + 8, xs[b + 1]);
                ya = q8_value(qw[b + 1], j, wd[b + 1]);
                yb = q8_value(qw[b + 1], j + 8, wd[b + 1]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = (c0[i] + c0[16 + i]) + (c1[i] + c1[16 + i]);
        asm volatile("" : "+v"(s));          // added here: left alone, the additions sink and both chains spill
        return s;
    };
    auto s4 = [&](int j) __attribute__((always_inline)) { f32x16 x = s8(j); x = x + s8(j + 4); asm volatile("" : "+v"(x)); return x; };
    auto s2 = [&](int j) __attribute__((always_inline)) { f32x16 x = s4(j); x = x + s4(j + 2); asm volatile("" : "+v"(x)); return x; };
    f32x16 s = s2(0);
    s = s + s2(1);
    // row of register i: token 8 (i / 4) + 4 (lane >> 5) + (i & 3); column: output lane & 31
    const int o = o0 + r;
    if (o >= a.d_out) return;
    char * d = reinterpret_cast<char *>(a.dst) + (size_t)h * a.d_nb2 + 4 * (size_t)o;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int t = t0 + 8 * (i >> 2) + 4 * kh + (i & 3);
        if (t < a.nt) *reinterpret_cast<float *>(d + (size_t)t * a.d_nb1) = s[i];
    }
}

// WKB over 32 tokens of one head: wave w of column group z takes 32-column blocks 4 z + w, + 4 Z, ...  The
// int32 dot of one Q8 block is one v_mfma_i32_32x32x32_i8 (exact), then acc = fma(wd * d16, sum,
// acc) over the blocks in order, the per-token kernel's operations bit for bit.
template <int NB>
__global__ __launch_bounds__(256) void wkb_q8_gemm_kernel(WkbArgs a) {
    typedef int i32x16 __attribute__((ext_vector_type(16)));
    __shared__ __attribute__((aligned(16))) char xq[GT * (NB * 32 + Q_PAD)];
    __shared__ __attribute__((aligned(16))) float xd[NB][GT];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 31, kh = lane >> 5;
    const int h = blockIdx.x, t0 = blockIdx.y * GT;
    quant_tokens<NB, true>(reinterpret_cast<const char *>(a.q) + (size_t)h * a.q_nb1, a.q_nb2, t0, a.nt, xq, xd);
    __syncthreads();
    i32x4 qx[NB];
    f32x4 xs[NB][4];                         // scales of this lane's 16 result rows (tokens)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        qx[b] = *reinterpret_cast<const i32x4 *>(xq + r * (NB * 32 + Q_PAD) + 32 * b + 16 * kh);
#pragma unroll
        for (int i = 0; i < 4; ++i) xs[b][i] = *reinterpret_cast<const f32x4 *>(&xd[b][8 * i + 4 * kh]);
    }
    for (int c0 = 128 * blockIdx.z + 32 * w; c0 < a.d_v; c0 += 128 * gridDim.z) {
        const int c = c0 + r;
        const uint8_t * wrow = a.wq + ((size_t)h * a.d_v + min(c, a.d_v - 1)) * (NB * 34);
        u32x4 qw[NB];
        float wd[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            qw[b] = q8_half_block(wrow, b, kh);
            wd[b] = f16_bits(*reinterpret_cast<const uint16_t *>(wrow + 34 * b));
        }
        f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            i32x16 s;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0;
            s = __builtin_amdgcn_mfma_i32_32x32x32_i8(qx[b], __builtin_bit_cast(i32x4, qw[b]), s, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = fmaf(wd[b] * xs[b][i >> 2][i & 3], (float)s[i], acc[i]);
        }
        if (c < a.d_v) {
            char * d = reinterpret_cast<char *>(a.dst) + (size_t)h * a.d_nb1 + 4 * (size_t)c;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int t = t0 + 8 * (i >> 2) + 4 * kh + (i & 3);
                if (t < a.nt) *reinterpret_cast<float *>(d + (size_t)t * a.d_nb2) = acc[i];
            }
        }
    }
}

// ---- PHASE 0, KV-write ----
// gemv: a workgroup per two output rows (m4-phase.cu:95-125).  The input is quantised once per workgroup,
// half a 32-value block per thread, into LDS; then a thread per (row, block): acc = (wd * d16) * sum, the
// butterfly per 32 blocks, and the 32-block partials summed in order.  The row's loads go out before
// the quantisation.  (A thread per block that quantised its own 32 values, a workgroup per row:
// 128-byte strides between lanes, and twice the work per thread before the first dot.)
template <int NBE>
__global__ __launch_bounds__(2 * NBE) void kvwrite_gemv_kernel(KvWriteArgs a) {
    // the reference's product (wd * d16) * sum and the butterfly's adds are separate statements;
    // without this the compiler fuses the first add with the product (one rounding instead of two)
#pragma clang fp contract(off)
    static_assert(NBE % 32 == 0 && 2 * NBE <= 1024, "whole 32-block groups");
    __shared__ __attribute__((aligned(16))) uint32_t xq[NBE * 8];
    __shared__ float xd[NBE];
    __shared__ float sv[2][NBE / 32];
    const int tid = threadIdx.x;
    const int r = tid >= NBE ? 1 : 0, blk = tid - r * NBE;
    const int o = 2 * blockIdx.x + r;        // n_out is a multiple of 32
    // the block's 34 bytes: 2-byte aligned; read the 9 dwords around it and realign
    const size_t boff = ((size_t)o * (NBE * 34)) + 34 * (size_t)blk;
    const uint32_t * bw = reinterpret_cast<const uint32_t *>(a.w + (boff & ~(size_t)3));
    const int sh = (int)(boff & 3);          // 0 or 2
    // (at sh = 0 the last two bytes of the 9th dword are the next block's: read only the 16 bits
    // that belong to this one, so the last block of the tensor reads nothing past its end)
    uint32_t D[9];
#pragma unroll
    for (int i = 0; i < 8; ++i) D[i] = bw[i];
    D[8] = sh ? bw[8] : (uint32_t)*reinterpret_cast<const uint16_t *>(bw + 8);
    // half block tid of the input
    {
        F4u x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const F4u *>(a.cur + 16 * tid + 4 * i);
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(x[i >> 2].v[i & 3]));
        amax = fmaxf(amax, dpp_xor<1>(amax));
        const float d = amax / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        u32x4 q;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t wv = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) wv |= ((uint32_t)(uint8_t)(int8_t)(int)roundf(x[j].v[e] * id)) << (8 * e);
            q[j] = wv;
        }
        *reinterpret_cast<u32x4 *>(xq + 4 * tid) = q;
        if ((tid & 1) == 0) xd[tid >> 1] = round_to_f16(d);
    }
    __syncthreads();
    const float wd = f16_bits((D[0] >> (8 * sh)) & 0xffffu);
    const u32x4 q0 = *reinterpret_cast<const u32x4 *>(xq + 8 * blk), q1 = *reinterpret_cast<const u32x4 *>(xq + 8 * blk + 4);
    int s = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t qw = sh ? D[j + 1] : __builtin_amdgcn_alignbyte(D[j + 1], D[j], 2);
        const uint32_t qx = j < 4 ? q0[j & 3] : q1[j & 3];
        s = __builtin_amdgcn_sdot4((int)qw, (int)qx, s, false);
    }
    float acc = (wd * xd[blk]) * (float)s;
    acc = half_wave_sum(acc);
    if ((blk & 31) == 0) sv[r][blk >> 5] = acc;
    __syncthreads();
    if (blk == 0) {
        float total = sv[r][0];
#pragma unroll
        for (int g = 1; g < NBE / 32; ++g) total += sv[r][g];
        a.dst[o] = total;
    }
}

// tail: one workgroup of n_out threads (m4-phase.cu:130-200).  Every thread reads its inputs
// (its row of the gemv output, and for a rope row both of its pair), the squares of the latent
// rows are reduced (butterfly per 32 rows, then the partials in order), and each thread writes its
// final value to dst and, as f16, to cache row kidx -- read on the device from the graph's
// tensors; a row outside [0, n_kv) is not written (the reference trusts the engine; this
// implementation refuses to scatter out of bounds).  With a Q8_0 cache (kc_q8) each 32-thread
// half-wavefront holds one block of the row and stores it as ggml's f32 -> q8_0 copy does
// (quantize_row_q8_0_ref, ggml-quants.c:276-299): d = amax / 127, q = roundf(x * (1 / d)), the
// f16 scale by the block's first lane, one int8 per lane.  n_out is a multiple of 32, so a
// half-wavefront is either all inside the row or all past it.
__global__ __launch_bounds__(1024) void kvwrite_tail_kernel(KvWriteArgs a) {
    __shared__ float sred[32];
    const int tid = threadIdx.x;
    const int n_out = a.d_lat + a.n_rope;
    const int64_t row = a.kidx[0];
    const int pos = a.pos[0];
    const bool lat = tid < a.d_lat;
    const bool rope = !lat && tid < n_out;
    const float v = tid < n_out ? a.dst[tid] : 0.0f;
    float x0 = 0.0f, x1 = 0.0f;
    const int p = (tid - a.d_lat) >> 1;     // the rope pair of a rope row
    if (rope) {
        x0 = a.dst[a.d_lat + 2 * p];
        x1 = a.dst[a.d_lat + 2 * p + 1];
    }
    const float sq = lat ? v * v : 0.0f;
    const float part = half_wave_sum(sq);
    if ((tid & 31) == 0) sred[tid >> 5] = part;
    __syncthreads();                         // (also: every input of dst has been read)
    float s = 0.0f;
    for (int g = 0; g < (n_out + 31) / 32; ++g) s += sred[g];
    float out = 0.0f;
    if (lat) {
        const float scale = rsqrtf(s / (float)a.d_lat + a.eps);
        out = scale * v * a.nw[tid];
    } else if (rope) {
        const float theta_extrap = (float)pos * powf(a.theta_scale, (float)p);
        float mscale = a.attn_factor;
        float theta = a.freq_scale * theta_extrap;
        if (a.ext_factor != 0.0f) {
            const float y = ((float)p - a.corr0) / fmaxf(0.001f, a.corr1 - a.corr0);
            const float ramp_mix = (1.0f - fminf(1.0f, fmaxf(0.0f, y))) * a.ext_factor;
            theta = theta * (1.0f - ramp_mix) + theta_extrap * ramp_mix;
            mscale *= 1.0f + 0.1f * logf(1.0f / a.freq_scale);
        }
        const float co = cosf(theta) * mscale, si = sinf(theta) * mscale;
        out = ((tid - a.d_lat) & 1) ? x0 * si + x1 * co : x0 * co - x1 * si;
    }
    if (a.kc_q8) {
        float d16;
        const int q = quant_lane<false>(out, d16);   // every lane takes part in the block max
        if (tid < n_out) {
            a.dst[tid] = out;
            if (row >= 0 && row < a.n_kv) {
                char * blk = reinterpret_cast<char *>(a.kcache) + (size_t)row * a.kc_nb1 + (size_t)(tid >> 5) * 34;
                if ((tid & 31) == 0) *reinterpret_cast<half_t *>(blk) = (half_t)d16;
                reinterpret_cast<int8_t *>(blk + 2)[tid & 31] = (int8_t)q;
            }
        }
        return;
    }
    if (tid < n_out) {
        a.dst[tid] = out;
        if (row >= 0 && row < a.n_kv)
            reinterpret_cast<half_t *>(reinterpret_cast<char *>(a.kcache) + (size_t)row * a.kc_nb1)[tid] = (half_t)out;
    }
}

}  // namespace

hipError_t launch_wkb_q8(const WkbArgs & a, hipStream_t stream) {
    if (wkb_q8_tiled(a)) {
        // few workgroups: the columns are split over them too
        const int tb = (a.nt + GT - 1) / GT;
        const dim3 grid(a.n_head, tb, a.n_head * tb < 256 && a.d_v <= 128 * 65535 ? (a.d_v + 127) / 128 : 1);
        if (a.d_n == 64) hipLaunchKernelGGL(wkb_q8_gemm_kernel<2>, grid, dim3(256), 0, stream, a);
        else if (a.d_n == 128) hipLaunchKernelGGL(wkb_q8_gemm_kernel<4>, grid, dim3(256), 0, stream, a);
        else return hipErrorInvalidValue;
        return hipGetLastError();
    }
    const dim3 grid(a.n_head, a.nt);
    if (a.d_n == 64) hipLaunchKernelGGL(wkb_q8_kernel<2>, grid, dim3(256), 0, stream, a);
    else if (a.d_n == 128) hipLaunchKernelGGL(wkb_q8_kernel<4>, grid, dim3(256), 0, stream, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_wvb_q8(const WvbArgs & a, hipStream_t stream) {
    if (wvb_tiled(a)) {
        const dim3 grid((a.nt + GT - 1) / GT, (a.d_out + 127) / 128, a.n_head);
        if (a.d_in == 256) hipLaunchKernelGGL(wvb_q8_gemm_kernel<8>, grid, dim3(256), 0, stream, a);
        else if (a.d_in == 512) hipLaunchKernelGGL(wvb_q8_gemm_kernel<16>, grid, dim3(256), 0, stream, a);
        else return hipErrorInvalidValue;
        return hipGetLastError();
    }
    const dim3 grid((a.d_out + 7) / 8, a.n_head, a.nt);
    if (a.d_in == 256) hipLaunchKernelGGL(wvb_q8_kernel<8>, grid, dim3(256), 0, stream, a);
    else if (a.d_in == 512) hipLaunchKernelGGL(wvb_q8_kernel<16>, grid, dim3(256), 0, stream, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_kvwrite(const KvWriteArgs & a, hipStream_t stream) {
    const int n_out = a.d_lat + a.n_rope;
    if (n_out > 1024) return hipErrorInvalidValue;
    if (a.n_embd == 4096) hipLaunchKernelGGL(kvwrite_gemv_kernel<128>, dim3(n_out / 2), dim3(256), 0, stream, a);
    else if (a.n_embd == 7168) hipLaunchKernelGGL(kvwrite_gemv_kernel<224>, dim3(n_out / 2), dim3(448), 0, stream, a);
    else return hipErrorInvalidValue;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kvwrite_tail_kernel, dim3(1), dim3((n_out + 63) / 64 * 64), 0, stream, a);
    return hipGetLastError();
}

}  // namespace mla
