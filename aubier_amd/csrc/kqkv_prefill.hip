// kqkv_prefill.hip -- GGML_OP_M4_KQKV for several query tokens (chunked prefill), on MFMA.
//
// The op of patches/ggml-m4/m4-kqkv.cu:340-378 (which the reference only runs for one token) for
// nt >= 16 tokens: out[h, t] = softmax_j(kq_scale q[t, h] . K[j] + mask[t, j]) . V[j] over the
// cache.  With many tokens the work is a dense contraction (config 5: 285 GFLOP over a 9.4 MB
// cache), so the design is MFMA-bound rather than HBM-bound:
//   * One workgroup per (split, 32-head group, 4 tokens); wave w owns token 4 z + w with all 32
//     heads: its q fragments (144 VGPRs, loaded once), its online softmax and its o^T for all D_v
//     columns (16 accumulator tiles in AGPRs).  No state crosses waves, so each finishes its token
//     on its own.
//   * The four waves share every 64-key tile: each streams one 16-key slice of it into a two-stage
//     LDS ring (decode_common.h layout, cached DMA: the cache is re-read by every token group and
//     stays in L2 / MALL) plus its own token's 64 mask values, and then every wave runs all four
//     slices -- 4 tokens x 32 heads share each K / V byte read from LDS.  One workgroup barrier
//     per tile; the next tile's DMA goes out one instruction per fourth Q.K^T step.
//   * Per pair of slices (32 keys): S^T = K . Q^T (32 keys x 32 heads, v_mfma_f32_32x32x16_f16, the
//     accumulator in VGPRs: the output tiles fill the AGPRs), scores with the token's mask, a lazily
//     moved reference max (P = exp2(s - m) <= 2^15; the move test on each lane's own maximum), then
//     o^T += V^T . P^T (v_mfma_f32_32x32x16_f16, V^T by ds_read_b64_tr_b16).  A lane of S^T holds 16
//     scores of one head, which are P.V's operand as they lie (the k order of that MFMA is free as long
//     as V^T is read in the same one): no lane exchange, and conflict-free transpose reads.  Slice 1's
//     exponentials and the sums of P run between slice 0's P.V MFMAs.  l is summed from the same f16
//     P values.  q enters as f16, where ggml-cpu's mul_mat rounds it; P enters as f16 too, but
//     UNNORMALISED (exp2 of the score minus the lazy reference max, <= 2^15), where ggml-cpu rounds
//     the normalised softmax output -- at long context the latter is subnormal in f16, so the two
//     differ by more than one rounding (this kernel is the closer of the two to exact arithmetic).
//   * The loop runs over the tiles that hold a live key of the workgroup's tokens (live_keys).
// Measured on the MI355X, D_k 576, 1,024 tokens x 32 heads in one split, no mask: 4,096 keys 262 us =
// 1.11 PFLOP/s (287 us with one slice at a time and serial reads of the mask row), 64 keys 26 us
// (28).  A tile takes 2.9 us of its 1.8 us of MFMA with few workgroups or with all-zero operands and
// 3.9 us with ordinary ones on all 256 CUs, where the clock drops: at full load the kernel is bound
// by power, at a rate near the card's large f16 matrix product (1.17 PFLOP/s).  At 320: 157 us (197).
//
// Grid = (n_split, ceil(H/32), ceil(nt/4)), 256 threads.  Output as the decode kernels: partial
// blocks [group][token][split] (mla_kernels.h) for the merge, or o/l in f32 to dst with one split.
#include "prefill_pass.h"

namespace mla {

namespace {

using namespace decode;

template <int DK, int DV>
__global__ __launch_bounds__(NTHR, 1) void kqkv_prefill_f16_kernel(DecodeArgs a) {
    __shared__ __attribute__((aligned(16))) char ring[SliceGeom<DK>::RING];          // [stage][wave] K rows + mask
    __shared__ int live_of[NWAVE][2];
    // the last token groups, which see the most keys under a causal mask, start first
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t_w = ((int)gridDim.z - 1 - (int)blockIdx.z) * NWAVE + w;
    prefill_pass<DK, DV>(a, t_w, t_w < a.nt, ring, live_of);
}

}  // namespace

template <int DK, int DV>
static hipError_t launch_prefill(const DecodeArgs & a, int n_hgroups, hipStream_t stream) {
    dim3 grid(a.n_split, n_hgroups, (a.nt + NWAVE - 1) / NWAVE);
    hipLaunchKernelGGL((kqkv_prefill_f16_kernel<DK, DV>), grid, dim3(NTHR), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_kqkv_prefill_f16(int dk, int dv, const DecodeArgs & a, hipStream_t stream) {
    const int n_hgroups = (a.n_head + HG - 1) / HG;
    if (dk == 576 && dv == 512) return launch_prefill<576, 512>(a, n_hgroups, stream);
    if (dk == 320 && dv == 256) return launch_prefill<320, 256>(a, n_hgroups, stream);
    return hipErrorInvalidValue;
}

}  // namespace mla
