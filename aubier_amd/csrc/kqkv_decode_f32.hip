// kqkv_decode_f32.hip -- split-K MLA attention over an f32 latent+rope KV cache, f32 end to end, on the
// f32 matrix cores, for the two MLA geometries (the VALU kernel of kqkv_generic.hip keeps the others).
//
// The VALU kernel runs one workgroup per (split, head): every head reads the whole cache again, 32 x
// 9.4 MB through the L2s for 4,096 keys.  Here a workgroup takes 16 heads, so a cache byte is read
// H / 16 times, and Q.K^T and P.V are v_mfma_f32_16x16x4_f32 (f32 products and sums, as ggml-cpu's F32
// mul_mat; 256 FLOP per cycle and CU, twice the VALU's rate without its operand traffic).
//   * A split is a run of 16-key granules (GRAN_KEYS, as the VALU kernel), walked in 32-key tiles
//     clipped to the split.  The tile's rows and its mask values stream into a two-stage LDS ring by
//     LDS DMA, whole lines, 16-byte chunk c of row r at slot c ^ (r & 15): the operand reads of Q.K^T
//     (16 rows at one chunk) and of P.V (256 bytes of a row) touch every bank once.
//   * The k order of an MFMA is free as long as both operands agree, so every operand comes as 16-byte
//     reads: Q.K^T step (s, e) takes d = 16 s + 4 g + e (g = lane >> 4), P.V step st takes keys 8 g + st
//     and, for element e of the chunk a lane read, its own set of columns.
//   * Q.K^T: wave w takes keys 16 (w & 1) .. +15 and half w >> 1 of the row's d (its q, 72 VGPRs, is
//     loaded once); the halves meet through LDS.  Every wave then holds the tile's scores, 8 keys of
//     head lane & 15 per lane, and runs the online softmax for itself.  P.V: wave w owns a quarter
//     of the columns; P is its operand as it lies.
// Grid = (n_split, ceil(H/16), nt), 256 threads.  Output: the f32 partial records of mla_kernels.h, or
// o / l to dst with one split.
// Measured (partial + merge, one token, 32 heads, D_k 576, VALU kernel before): 1,024 keys 15.5 -> 12.2 us,
// 4,096 44.5 -> 16.2, 8,192 89.7 -> 19.0; error against float64 4.2e-7 -> 3.4e-7 at 1,024 keys, 4.2e-7 ->
// 2.9e-7 at 4,096.  Bound: for a decode step the launch, one tile's latency and the records (66 KB per split and 32
// heads, written here and read by the merge); from some 30,000 keys the f32 MFMAs.
#include "mla_common.h"
#include "mla_kernels.h"

namespace mla {

namespace {

constexpr int FTK = F32_TILE_KEYS;       // keys per tile
constexpr int FHG = F32_HEADS;           // heads per workgroup
static_assert(FTK == 32 && FHG == 16, "two key tiles of 16, 16 lanes of heads");
constexpr int SPITCH = FTK + 4;          // score exchange row pitch (floats)

template <int DK>
struct F32Geom {
    static constexpr int CH = DK / 4;                        // 16-byte chunks per row
    static constexpr int ROWS = FTK * CH * 16;               // bytes of a tile's rows
    static constexpr int STAGE = ROWS + 4 * 256;             // + a mask slot per wave
    static constexpr int NI = FTK / 4 * CH / 64;             // DMA instructions per wave: its 8 rows
    static constexpr int QS = DK / 32;                       // 16-d steps of half a row
    static_assert(CH % 16 == 0 && FTK / 4 * CH % 64 == 0 && DK % 32 == 0, "whole swizzle blocks, whole instructions");
};

template <int DK>
struct F32Lds {
    __attribute__((aligned(16))) char ring[2][F32Geom<DK>::STAGE];
    __attribute__((aligned(16))) float sx[2][FHG][SPITCH];   // score halves [d half][head][key]
};

template <int DK, int DV>
__global__ __launch_bounds__(256, 1) void kqkv_decode_f32_kernel(DecodeArgs a) {
    using G = F32Geom<DK>;
    constexpr int NT = DV / 4 / 64;                          // 64-column groups per wave
    static_assert(DV % 256 == 0 && DV <= DK, "geometry");
    __shared__ F32Lds<DK> sh;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j16 = lane & 15, g = lane >> 4;
    const int sp = blockIdx.x, t = blockIdx.z;
    const int h = blockIdx.y * FHG + j16;                    // this lane's head

    // the split's keys [k0, k1)
    const int n_gran = (a.n_kv + GRAN_KEYS - 1) / GRAN_KEYS;
    const int base_g = n_gran / a.n_split, rem_g = n_gran % a.n_split;
    const int k0 = (sp * base_g + min(sp, rem_g)) * GRAN_KEYS;
    const int k1 = min(k0 + (base_g + (sp < rem_g ? 1 : 0)) * GRAN_KEYS, a.n_kv);
    const int n_tile = (k1 - k0 + FTK - 1) / FTK;            // 0 for a split without keys

    // this wave's q: head j16, d = DK / 2 (w >> 1) + 16 s + 4 g .. +3
    f32x4 q[G::QS];
    {
        const char * row = reinterpret_cast<const char *>(a.q) + (size_t)t * a.q_nb2 + (size_t)min(h, a.n_head - 1) * a.q_nb1 +
                           4 * (DK / 2 * (w >> 1) + 4 * g);
#pragma unroll
        for (int s = 0; s < G::QS; ++s) q[s] = *reinterpret_cast<const f32x4 *>(row + 64 * s);
    }
    // DMA plan: wave w fetches rows 8 w .. 8 w + 7 of the tile, slot p = 64 i + lane of its 8 CH
    uint32_t voff[G::NI];
#pragma unroll
    for (int i = 0; i < G::NI; ++i) {
        const int p = 64 * i + lane;
        const int r = FTK / 4 * w + p / G::CH;
        voff[i] = (uint32_t)(r * a.kc_nb1) + 16u * (uint32_t)((p % G::CH) ^ (r & 15));
    }
    const float * mrow = a.mask ? reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.mask) + (size_t)t * a.mask_nb1) : a.q;
    // rows (and mask values) at or past the split's end come back as zeros
    auto dma = [&](int k) __attribute__((always_inline)) {
        const int key = k0 + FTK * k;
        const int left = min(k1 - key, FTK);                 // >= 1
        const i32x4 krs = make_rsrc(a.kc + (int64_t)key * a.kc_nb1, (uint32_t)((int64_t)(left - 1) * a.kc_nb1 + DK * 4));
        const i32x4 mrs = make_rsrc(mrow + key, a.mask ? (uint32_t)left * 4u : 0u);
        const uint32_t sb = lds_addr(sh.ring[k & 1]);
#pragma unroll
        for (int i = 0; i < G::NI; ++i) dma16_nt(krs, voff[i], 0u, sb + (uint32_t)((FTK / 4 * w * G::CH + 64 * i) * 16));
        dma4(mrs, 4u * (uint32_t)(lane & 31), 0u, sb + (uint32_t)(G::ROWS + 256 * w));
    };

    float m_run = -INFINITY, l_run = 0.0f;                   // head j16; l of this lane's keys only
    f32x4 o[NT][4];                                          // [T][e][r]: column DV/4 w + 64 T + 16 r + 4 g + e of head j16
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[T][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    if (n_tile > 0) dma(0);
    for (int k = 0; k < n_tile; ++k) {
        if (k + 1 < n_tile) {
            if (k > 0) __syncthreads();      // every wave is past tile k - 1, whose stage tile k + 1 takes
            dma(k + 1);
            wait_vm<G::NI + 1>();            // this wave's part of tile k has landed
        } else {
            wait_vm<0>();
        }
        __syncthreads();
        const char * st = sh.ring[k & 1];
        // ---- S^T = K . Q^T of 16 keys over half of d: C row = key 4 g + r, C col = head j16 ----
        {
            const int kt = w & 1, dh = w >> 1;
            const char * row = st + (16 * kt + j16) * (G::CH * 16);
            // eight chains: with the halves, sums of D_k / 16 products each (the VALU kernel's hold D_k / 8;
            // two chains of D_k / 4 left results 15% further from float64 than it, these are nearer)
            f32x4 c[2][4];
#pragma unroll
            for (int e = 0; e < 8; ++e) c[e >> 2][e & 3] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < G::QS; ++s) {
                const f32x4 kv = *reinterpret_cast<const f32x4 *>(row + 16 * ((G::CH / 2 * dh + 4 * s + g) ^ j16));
#pragma unroll
                for (int e = 0; e < 4; ++e) c[s & 1][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[e], q[s][e], c[s & 1][e], 0, 0, 0);
            }
            *reinterpret_cast<f32x4 *>(&sh.sx[dh][j16][16 * kt + 4 * g]) =
                ((c[0][0] + c[1][0]) + (c[0][1] + c[1][1])) + ((c[0][2] + c[1][2]) + (c[0][3] + c[1][3]));
        }
        __syncthreads();
        // ---- scores of keys 8 g + i, online softmax (every wave the same values) ----
        float p[8];
        {
            const float * mk = reinterpret_cast<const float *>(st + G::ROWS + 256 * w) + 8 * g;
            const int left = k1 - (k0 + FTK * k) - 8 * g;    // this lane's keys inside the split
            float mx = -INFINITY;
#pragma unroll
            for (int i4 = 0; i4 < 2; ++i4) {
                const f32x4 sa = *reinterpret_cast<const f32x4 *>(&sh.sx[0][j16][8 * g + 4 * i4]);
                const f32x4 sb = *reinterpret_cast<const f32x4 *>(&sh.sx[1][j16][8 * g + 4 * i4]);
                const f32x4 m4 = *reinterpret_cast<const f32x4 *>(mk + 4 * i4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 4 * i4 + e;
                    p[i] = i < left ? (sa[e] + sb[e]) * a.scale_log2 + m4[e] * LOG2E : -INFINITY;
                    mx = fmaxf(mx, p[i]);
                }
            }
            mx = fmaxf(m_run, rows4_max(mx));
            const float alpha = exp2_unless(m_run == -INFINITY, m_run - mx);
            m_run = mx;
            l_run *= alpha;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                p[i] = exp2_unless(p[i] == -INFINITY, p[i] - mx);
                l_run += p[i];
            }
#pragma unroll
            for (int T = 0; T < NT; ++T)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[T][e] *= alpha;
        }
        // ---- O^T += V^T . P^T over the tile's 32 keys: step i takes keys 8 g + i ----
        // lane j16 reads chunk 4 (j16 & 3) + (j16 >> 2) of a 64-column group, so that a lane's results lie
        // next to its neighbours' (64-byte runs in the record)
        {
            const int cp = 4 * (j16 & 3) + (j16 >> 2);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int sw = 8 * (g & 1) + i;              // (8 g + i) & 15
                const char * row = st + (8 * g + i) * (G::CH * 16) + 16 * (cp ^ sw) + DV * w;
#pragma unroll
                for (int T = 0; T < NT; ++T) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(row + 256 * T);
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[T][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], p[i], o[T][e], 0, 0, 0);
                }
            }
        }
    }

    float ev, od;
    rows_pair16(l_run, ev, od);
    const float L = halves_sum(ev + od);
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    if (h >= a.n_head) return;
    float * d;
    if (a.dst != nullptr) {
        d = a.dst + ((size_t)h * a.nt + t) * DV;
    } else {
        const int hh = h % PART_HEADS;
        char * rec = part_record(a.part, h / PART_HEADS, a.nt, t, a.n_split, DV, 4);
        if (w == 0 && g == 0) {
            float lr = L;
            if (m_run == -INFINITY && L != L && !any_live_key(a, t, k0, k1)) lr = 0.0f;
            *reinterpret_cast<f32x2 *>(rec + part_ml_off(a.n_split, hh, sp)) = f32x2{(m_run == -INFINITY) ? -INFINITY : m_run * LN2, lr};
        }
        if (m_run == -INFINITY) return;                      // no live key: the merge never reads this o
        d = reinterpret_cast<float *>(rec + part_o_off(a.n_split, sp, DV, 4)) + (size_t)hh * DV;
    }
    d += DV / 4 * w + 4 * g;
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4 *>(d + 64 * T + 16 * r) = f32x4{o[T][0][r], o[T][1][r], o[T][2][r], o[T][3][r]} * inv;
}

}  // namespace

hipError_t launch_kqkv_decode_f32(int dk, int dv, const DecodeArgs & a, hipStream_t stream) {
    const dim3 grid(a.n_split, (a.n_head + FHG - 1) / FHG, a.nt);
    if (dk == 576 && dv == 512) hipLaunchKernelGGL((kqkv_decode_f32_kernel<576, 512>), grid, dim3(256), 0, stream, a);
    else if (dk == 320 && dv == 256) hipLaunchKernelGGL((kqkv_decode_f32_kernel<320, 256>), grid, dim3(256), 0, stream, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace mla
