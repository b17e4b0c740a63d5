// prefill_pass.h -- the pass of four tokens over one split of an f16 cache, a wave per token, on MFMA:
// the prefill kernel's body (kqkv_prefill.hip describes the design), and what the decode kernel runs for
// rows that share a split (kqkv_decode.hip).
#pragma once

#include "decode_common.h"

namespace mla {
namespace decode {

template <int DK, int DV>
struct PrefillCfg {
    using G = SliceGeom<DK>;
    static_assert(DV % 128 == 0 && DV <= DK, "geometry");
    static constexpr int NB = DV / 32;                  // 32-column o^T tiles per wave
    static constexpr int OPITCH = DV * 2 + 16;          // f16 output staging row pitch (bytes)
    static constexpr int CPR = DV / 8;                  // 16-byte output chunks per head row
    static_assert(NWAVE * HG * OPITCH <= G::RING, "the output staging fits the ring");
    static_assert(CPR % 2 == 0 && NB - 1 < 64, "layout");
};

// Split blockIdx.x, head group blockIdx.y, wave w's token t_w (token_live: there is one; the others mirror
// the last token and write nothing).  `ring`: G::RING bytes of LDS, 16-byte aligned; the caller keeps its
// next use of ring and live_of behind a barrier.
template <int DK, int DV>
__device__ __forceinline__ void prefill_pass(const DecodeArgs & a, int t_w, bool token_live, char * ring, int (&live_of)[NWAVE][2]) {
    using G = SliceGeom<DK>;
    using C = PrefillCfg<DK, DV>;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sp = blockIdx.x;
    const int hg0 = blockIdx.y * HG;
    const int t = min(t_w, a.nt - 1);                // (a wave past the last token mirrors it, unused)

    SliceStream<DK> ss(a, sp, t, w, lds_addr(ring), lane);
    ss.mvoff = 4u * (uint32_t)lane;                  // the mask slot holds this token's 64 keys of the tile
    const int n_my = ss.n_my;
    // DMA of tile k into stage s: this wave's 16-key slice of K rows (cached policy: every token
    // group re-reads the cache) and this wave's token's mask over the tile's 64 keys (zeros past
    // n_kv or without a mask)
    auto plan = [&](int s, int k) {
        SliceDma d = ss.plan(s, k);
        const int tile = min(ss.t0 + min(k, n_my - 1), ss.n_tiles - 1);
        const int mleft = a.n_kv - tile * TK;
        d.mrs = make_rsrc(ss.mrow + tile * TK, (ss.has_mask && mleft > 0) ? (uint32_t)mleft * 4u : 0u);
        return d;
    };
    // The tiles of the split that hold a live key (mask > -inf) of this wave's token, [ka_w, kz_w), and of
    // any of the workgroup's, [ka, kz): the loop runs over the latter (a causal chunk's first tokens see
    // few of the window's tiles; rows over per-sequence regions one run of them), and a wave computes
    // only in its own.  A workgroup with no live key records empty splits and leaves before any DMA.
    int first, last;
    live_keys(ss.has_mask ? ss.mrow : nullptr, ss.t0 * TK, token_live ? min((ss.t0 + n_my) * TK, a.n_kv) : 0, lane, first, last);
    const bool live_w = first <= last;
    const int ka_w = live_w ? first / TK - ss.t0 : 0, kz_w = live_w ? last / TK - ss.t0 + 1 : 0;
    if (lane == 0) {
        live_of[w][0] = live_w ? ka_w : n_my;
        live_of[w][1] = kz_w;
    }
    __syncthreads();
    const int ka = min(min(live_of[0][0], live_of[1][0]), min(live_of[2][0], live_of[3][0]));
    const int kz = max(max(live_of[0][1], live_of[1][1]), max(live_of[2][1], live_of[3][1]));
    if (ka >= kz && a.dst == nullptr) {
        if (token_live) write_empty_pairs(a, blockIdx.y, t, sp, DV, lane);
        return;
    }
    {
        const SliceDma d0 = plan(ka & 1, ka);
#pragma unroll
        for (int i = 0; i <= G::DMA_N; ++i) ss.template put<false>(d0, i);
    }

    // ---- q fragments of this wave's token: qf[st] = head lane & 31, d = 16 st + 8 (lane >> 5) .. +7 ----
    // Read in batches of QB fragments, each batch's loads issued before the one ahead of it is
    // converted: a batch at a time, every batch paid the memory latency.
    const int hl = lane & 31, hi = lane >> 5;
    half8 qf[DK / 16];
    {
        constexpr int QB = DK / 16 % 6 == 0 ? 6 : 5;
        constexpr int NBT = DK / 16 / QB;
        static_assert(NBT * QB == DK / 16, "whole batches");
        const bool hv = hg0 + hl < a.n_head;
        const char * row = reinterpret_cast<const char *>(a.q) + (size_t)t * a.q_nb2 +
                           (size_t)min(hg0 + hl, a.n_head - 1) * a.q_nb1 + 32 * hi;
        f32x4 x[2][QB][2];
        auto load = [&](int i, f32x4 (&xb)[QB][2]) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                xb[b][0] = *reinterpret_cast<const f32x4 *>(row + 64 * (QB * i + b));
                xb[b][1] = *reinterpret_cast<const f32x4 *>(row + 64 * (QB * i + b) + 16);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        load(0, x[0]);
#pragma unroll
        for (int i = 0; i < NBT; ++i) {
            if (i + 1 < NBT) load(i + 1, x[(i + 1) & 1]);
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                const f32x4 (&y)[2] = x[i & 1][b];
                half8 hq = {to_half(y[0][0]), to_half(y[0][1]), to_half(y[0][2]), to_half(y[0][3]),
                            to_half(y[1][0]), to_half(y[1][1]), to_half(y[1][2]), to_half(y[1][3])};
                if (!hv) hq = half8{0, 0, 0, 0, 0, 0, 0, 0};
                asm volatile("" : "+v"(hq));         // keep the f16 fragment (not the f32 values) live
                qf[QB * i + b] = hq;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- per-wave state ----
    float m_run = M_NONE;                    // head hl, log2 units
    float l_acc = 0.0f;                      // head hl, this lane's half of the keys
    f32x16 o[C::NB];                         // o^T tile i: C row = column 32 i + 8 (r / 4) + 4 hi + (r & 3), C col = head hl
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.0f;
    const PairPvAddr pv(lane);

    for (int k = ka; k < kz; ++k) {
        wait_vm<0>();                        // this wave's slot of tile k (and its mask row) has landed
        __syncthreads();                     // all four have; every wave is done with tile k - 1
        const bool pf = k + 1 < kz;
        const SliceDma dn = plan((k + 1) & 1, k + 1);
        const int par = k & 1;
        const int key_t = (ss.t0 + k) * TK;
        const char * mkb = ring + ss.stage_off(par, w) + G::ROWS_BYTES;    // this token's mask, 64 keys
        if (k < ka_w || k >= kz_w) {         // only this wave's slice of the next tile
            if (pf) {
#pragma unroll
                for (int i = 0; i <= G::DMA_N; ++i) ss.template put<false>(dn, i);
            }
            continue;
        }
        // the first pair's first Q.K^T operands (the second's: during the P.V before)
        half8 abuf[QPF_LANDED];
        qk_operands<DK>(ring + ss.stage_off(par, 0), lane, abuf);
#pragma unroll 1
        for (int kp = 0; kp < NWAVE / 2; ++kp) {
            const char * sb = ring + ss.stage_off(par, 2 * kp);
            f32x16 s;
            // tile k + 1's DMA, one instruction per fourth Q.K^T step (row blocks DMA_N / 2 * kp + st / 4)
            // and the mask slot after the second pair's last step: the CU's 76 KB of DMA per tile,
            // issued at once, held the issuing waves ~450 cycles
            if (pf) {
                qk_pair_landed<DK>(sb, lane, qf, abuf, s, [&](int st) {
                    constexpr int HALF = G::DMA_N / 2;
                    static_assert(G::DMA_N % 2 == 0 && DK / 16 == 2 * G::DMA_N, "two pairs of slices of row blocks");
                    if ((st & 3) == 0) ss.template put<false>(dn, HALF * kp + st / 4);
                    else if (st == DK / 16 - 1 && kp == 1) ss.template put<false>(dn, G::DMA_N);
                });
            } else {
                qk_pair_landed<DK>(sb, lane, qf, abuf, s, [](int) {});
            }
            // the pair's mask values of this lane's keys and the first V^T operands of P.V, read ahead so
            // that their latency passes under the scores and the softmax
            f32x4 mk[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) mk[j] = *reinterpret_cast<const f32x4 *>(mkb + 4 * (32 * kp + 8 * j + 4 * hi));
            constexpr int VPF = 3;
            half8 vb[VPF];
#pragma unroll
            for (int i = 0; i < VPF; ++i) vb[i] = pv.load(sb, i);
            __builtin_amdgcn_sched_barrier(0);
            // scores in log2 units; a key past n_kv (its K row and mask read as zeros) takes -inf
            const int key0 = key_t + 32 * kp + 4 * hi;
            if (key_t + TK > a.n_kv) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (key0 + 8 * (r >> 2) + (r & 3) >= a.n_kv) mk[r >> 2][r & 3] = -INFINITY;
            }
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = s[r] * a.scale_log2 + mk[r >> 2][r & 3] * LOG2E;
                mx = fmaxf(mx, s[r]);
            }
            if (__builtin_amdgcn_ballot_w64(ref_moves(m_run, mx)) != 0) {
                // rare: move the reference to the head's max over the pair, rescale
                float lo, up;
                halves_pair(mx, lo, up);
                mx = fmaxf(lo, up);
                const bool mv = ref_moves(m_run, mx);
                // a head with no live key so far holds zeros: nothing to rescale
                const bool scale = mv && m_run != M_NONE;
                const float al = scale ? exp2_fast(m_run - (mx - REF_DROP)) : 1.0f;
                m_run = mv ? mx - REF_DROP : m_run;
                if (__builtin_amdgcn_ballot_w64(scale) != 0) {
                    l_acc *= al;
                    // in place on the accumulator registers (kept in AGPRs); the s_nops cover the
                    // MFMA -> VALU read distance
                    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
                    for (int i = 0; i < C::NB; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            float tmp;
                            asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
                                         : "+a"(o[i][r]), "=&v"(tmp) : "v"(al));
                        }
                    asm volatile("s_nop 7" ::: "memory");
                }
            }
            // P^T operands of the two slices, P.V of the slices in turn; slice 1's exponentials and the sums
            // of P run between slice 0's MFMAs (32 cycles each, which cover a few VALU instructions of
            // the same wave)
            half8 pt[2];
            auto put_p = [&](int j, int e0) __attribute__((always_inline)) {
#pragma unroll
                for (int e = e0; e < e0 + 4; ++e) pt[j][e] = to_half(exp2_fast(s[8 * j + e] - m_run));
            };
            put_p(0, 0);
            put_p(0, 4);
#pragma unroll
            for (int u = 0; u < 2 * C::NB; ++u) {
                const half8 va = vb[u % VPF];
                if (u + VPF < 2 * C::NB) vb[u % VPF] = pv.load(sb + G::STAGE * ((u + VPF) / C::NB), (u + VPF) % C::NB);
                o[u % C::NB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, pt[u / C::NB], o[u % C::NB], 0, 0, 0);
                if (u == 1) put_p(1, 0);
                if (u == 3) put_p(1, 4);
                if (u % C::NB < 4)
                    l_acc = __builtin_amdgcn_fdot2(half2{pt[u / C::NB][2 * (u % C::NB)], pt[u / C::NB][2 * (u % C::NB) + 1]}, ONE2, l_acc, false);
                if (u == C::NB + C::NB / 2 && kp + 1 < NWAVE / 2)       // the next pair's operands
                    qk_operands<DK>(ring + ss.stage_off(par, 2 * kp + 2), lane, abuf);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    wait_vm<0>();
    __syncthreads();                         // the ring becomes the output staging
    int tid_e;
    asm volatile("v_mov_b32 %0, %1" : "=v"(tid_e) : "v"(tid));
    const int lane_e = tid_e & 63;
    const float L = halves_sum(l_acc);         // head lane & 31, all keys of the split
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    if (!token_live) return;
    if (!live_w && a.dst == nullptr) {       // (with one split a token without a live key writes zeros below)
        write_empty_pairs(a, blockIdx.y, t, sp, DV, lane_e);
        return;
    }
    const int hi4 = 4 * (lane_e >> 5), hle = lane_e & 31;
    if (a.dst != nullptr) {                  // single split: o / l in f32 straight to dst
        const int h = hg0 + hle;
        if (h < a.n_head) {
            float * d = a.dst + ((size_t)h * a.nt + t) * DV + hi4;
#pragma unroll
            for (int i = 0; i < C::NB; ++i)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4)
                    *reinterpret_cast<f32x4 *>(d + 32 * i + 8 * q4) =
                        f32x4{o[i][4 * q4] * inv, o[i][4 * q4 + 1] * inv, o[i][4 * q4 + 2] * inv, o[i][4 * q4 + 3] * inv};
        }
        return;
    }
    char * rec = part_record(a.part, blockIdx.y, a.nt, t, a.n_split, DV, 2);
    char * blk = rec + part_o_off(a.n_split, sp, DV, 2);
    if (lane_e < HG) {
        *reinterpret_cast<f32x2 *>(rec + part_ml_off(a.n_split, lane_e, sp)) =
            f32x2{(m_run == M_NONE) ? -INFINITY : m_run * LN2, L};                   // m in natural-log units
    }
    // o / l in f16 through this wave's staging rows [32 heads][D_v], then 16-byte row chunks out
    char * stg = ring + w * HG * C::OPITCH;
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const half4 hv = {to_half(o[i][4 * q4] * inv), to_half(o[i][4 * q4 + 1] * inv), to_half(o[i][4 * q4 + 2] * inv),
                              to_half(o[i][4 * q4 + 3] * inv)};
            *reinterpret_cast<half4 *>(stg + hle * C::OPITCH + (32 * i + 8 * q4 + hi4) * 2) = hv;
        }
#pragma unroll
    for (int it = 0; it < C::CPR / 2; ++it) {
        const int q = 64 * it + lane_e;
        const int row = q / C::CPR, ch = q % C::CPR;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(stg + row * C::OPITCH + 16 * ch);
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(blk + ((size_t)row * DV + 8 * ch) * 2));
    }
}


}  // namespace decode
}  // namespace mla
