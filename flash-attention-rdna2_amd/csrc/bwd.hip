// bwd.hip — fable_attn_bwd and fable_attn_bwd_ds_bytes, the backward's C-ABI entry points:
// argument checks and dispatch to the per-width fp16/bf16 kernels (bwd_dNN.hip, kernels in
// bwd_kernel.hpp) and the fp32 kernels (bwd_f32.hip). Reference launcher:
// kernels/backward.hip:508-521.
#include "bwd_kernel.hpp"

namespace fa {

// fp16/bf16: every head dim that is a multiple of 8 up to 256 runs in the kernel of the next
// multiple of 32 (bwd_dNN.hip; the columns between are zero)
static int bwd_dispatch(const FableBwdParams& p, int dtype, hipStream_t st) {
  if (p.D <= 0 || p.D > 256 || p.D % 8)
    return fail(FA_ERR_HEADDIM, "fable_attn_bwd: head_dim=%d has no kernel (multiples of 8 up to 256)", p.D);
  switch (bwd_width(p.D)) {
    case 32: return launch_bwd_d32(p, dtype, st);
    case 64: return launch_bwd_d64(p, dtype, st);
    case 96: return launch_bwd_d96(p, dtype, st);
    case 128: return launch_bwd_d128(p, dtype, st);
    case 160: return launch_bwd_d160(p, dtype, st);
    case 192: return launch_bwd_d192(p, dtype, st);
    case 224: return launch_bwd_d224(p, dtype, st);
    default: return launch_bwd_d256(p, dtype, st);
  }
}

}  // namespace fa

namespace fa {
// A window at least as long as the sequences bounds nothing: dropping it keeps every mask bound
// in 32 bits (and the dS workspace layout the same for the size query and the launch).
static void normalize_windows(FableBwdParams& p) {
  if (p.win_left >= p.SK) p.win_left = -1;
  if (p.win_right >= p.SQ) p.win_right = -1;
}
}  // namespace fa

extern "C" int64_t fable_attn_bwd_ds_bytes(FableBwdParams p, int dtype) {
  if ((dtype != FA_F16 && dtype != FA_BF16) || p.D <= 0 || p.D % 8 || fa::bwd_width(p.D) > 256 || p.B <= 0 ||
      p.Hq <= 0)
    return 0;
  fa::normalize_windows(p);
  return fa::ds_bytes(p);
}

extern "C" int fable_attn_bwd(FableBwdParams p, int dtype, void* stream) {
  using namespace fa;
  if (!p.Q || !p.K || !p.V || !p.O || !p.dO || !p.dQ || !p.dK || !p.dV || !p.lse || !p.dsum)
    return fail(FA_ERR_ARG, "fable_attn_bwd: null pointer");
  if (p.Hq <= 0 || p.Hk <= 0 || p.Hq % p.Hk || p.gqa != p.Hq / p.Hk)
    return fail(FA_ERR_ARG, "fable_attn_bwd: Hq=%d Hk=%d gqa=%d", p.Hq, p.Hk, p.gqa);
  if (p.dropout && !(p.dropout_p >= 0.0f && p.dropout_p < 1.0f))
    return fail(FA_ERR_ARG, "fable_attn_bwd: dropout_p=%g", p.dropout_p);
  if ((p.cu_q == nullptr) != (p.cu_k == nullptr))
    return fail(FA_ERR_ARG, "fable_attn_bwd: cu_q and cu_k go together");
  if (p.B <= 0 || p.SQ < 0 || p.SK < 0) return FA_OK;  // empty ranges write zero gradients
  normalize_windows(p);
  if (!p.cu_q && p.lse_sb == 0 && p.lse_sh == 0) {  // dense [B,Hq,SQ] LSE / dsum
    p.lse_sh = p.SQ;
    p.lse_sb = (int64_t)p.Hq * p.SQ;
  }
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case FA_F16:
    case FA_BF16: return bwd_dispatch(p, dtype, st);
    case FA_F32: return launch_bwd_f32(p, st);
    default: return fail(FA_ERR_DTYPE, "fable_attn_bwd: dtype %d not implemented (fp16/bf16/fp32)", dtype);
  }
}

// ------------------------------------------------------------------ rows outside every sequence
namespace fa {

// Zeros in the rows of a packed tensor that no sequence uses: before cu[0], between a sequence's used
// rows and the next one's first, and from the last one's used rows to the end. The backward kernels
// write every row a sequence uses, so filling whole gradients first (three passes over them: 48 us for
// 25k rows of 32 + 2 x 8 heads, D 128) wrote nearly all of it twice. One launch for dQ, dK and dV:
// grid (workgroups, tensors), 16-byte stores. A buffer padded to a fixed size has its padding in the
// last gap (kTailParts workgroups), sequences cut by seqused in every gap (`slices` each): with 4 workgroups per
// gap 8 sequences of 512 rows ahead of 28k rows of padding took 15 us longer than the fill, now as long (47 us).
constexpr int kTailParts = 128, kUsedParts = 1024;
struct GapTensor {
  uint4* base;
  long long rows, row16;      // rows of the buffer, 16-byte units per row
  int most;                   // the longest sequence the caller named (the kernels' grids end there)
  const int *cu, *used;
};
__global__ __launch_bounds__(256) void zero_gaps_kernel(GapTensor a, GapTensor b, GapTensor c, int batch, int slices) {
  const GapTensor t = blockIdx.y == 0 ? a : (blockIdx.y == 1 ? b : c);
  const int g = min((int)blockIdx.x / slices, batch);   // gap g lies before sequence g (g = batch: after the last one)
  const long long part = (int)blockIdx.x - g * slices, parts = g < batch ? slices : kTailParts;
  long long r0 = 0, r1 = g < batch ? t.cu[g] : t.rows;
  if (g > 0) {
    const int s0 = t.cu[g - 1], len = t.cu[g] - s0;
    r0 = s0 + max(min(t.used ? min(len, t.used[g - 1]) : len, t.most), 0);
  }
  r0 = max(r0, 0ll) * t.row16;
  r1 = min(r1, t.rows) * t.row16;
  for (long long i = r0 + 256 * part + threadIdx.x; i < r1; i += 256 * parts) t.base[i] = uint4{0u, 0u, 0u, 0u};
}

}  // namespace fa

extern "C" int fable_attn_bwd_zero_gaps(FableBwdParams p, int dtype, int64_t total_q, int64_t total_k, void* stream) {
  using namespace fa;
  const int el = dtype == FA_F32 ? 4 : 2;
  // (arguments that fable_attn_bwd refuses are left for it to report)
  if (!p.dQ || !p.dK || !p.dV || !p.cu_q || !p.cu_k || p.D <= 0 || p.D % 8 || p.Hq <= 0 || p.Hk <= 0) return FA_OK;
  const long long nq = (long long)p.Hq * p.D * el, nk = (long long)p.Hk * p.D * el;
  if (((uintptr_t)p.dQ | (uintptr_t)p.dK | (uintptr_t)p.dV) & 15)
    return fail(FA_ERR_ARG, "fable_attn_bwd_zero_gaps: tensors are not 16-byte aligned");
  if (p.dqs.s != (int64_t)p.Hq * p.D || p.dks.s != (int64_t)p.Hk * p.D || p.dvs.s != (int64_t)p.Hk * p.D)
    return fail(FA_ERR_ARG, "fable_attn_bwd_zero_gaps: rows are not contiguous");
  if (p.B < 0) return FA_OK;
  // (with a negative length fable_attn_bwd writes nothing)
  const int mq = p.SQ < 0 || p.SK < 0 ? 0 : p.SQ, mk = p.SQ < 0 || p.SK < 0 ? 0 : p.SK;
  int slices = 1;
  if ((p.seqused_q || p.seqused_k) && p.B < kUsedParts) slices = kUsedParts / (p.B > 8 ? p.B : 8);
  hipLaunchKernelGGL(zero_gaps_kernel, dim3(p.B * slices + kTailParts, 3), dim3(256), 0, (hipStream_t)stream,
                     GapTensor{(uint4*)p.dQ, total_q, nq / 16, mq, p.cu_q, p.seqused_q},
                     GapTensor{(uint4*)p.dK, total_k, nk / 16, mk, p.cu_k, p.seqused_k},
                     GapTensor{(uint4*)p.dV, total_k, nk / 16, mk, p.cu_k, p.seqused_k}, p.B, slices);
  return launch_status("fable_attn_bwd_zero_gaps");
}
