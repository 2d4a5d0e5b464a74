// fwd.hip — the forward's C-ABI entry points (fable_attn_fwd, fable_attn_fwd_ws and the
// workspace query): argument checks and dispatch to the per-width fp16/bf16 kernels
// (fwd_d32.hip .. fwd_d256.hip, kernel in fwd_kernel.hpp) and the fp32 kernels (fwd_f32.hip);
// the merge of a key-split forward's partials. Reference launcher: kernels/fa_forward.hip:424-451.
#include <type_traits>

#include "attn_device.hpp"
#include "fwd_common.hpp"
#include "status.hpp"

namespace fa {

// fp16/bf16: every head dim that is a multiple of 8 up to 256 runs in the kernel of the next
// multiple of 32 (the columns between are zero: at most 24 of them, <= 1.75x the MFMA work at
// head dim 8, <= 1.1x from 80 up)
static int dispatch_hd(const FableFwdParams& p, int dtype, hipStream_t st, FwdWs& ws) {
  if (p.HD <= 0 || p.HD > 256 || p.HD % 8)
    return fail(FA_ERR_HEADDIM, "fable_attn_fwd: head_dim=%d has no kernel (multiples of 8 up to 256)", p.HD);
  switch ((p.HD + 31) / 32) {
    case 1: return launch_fwd_d32(p, dtype, st, ws);
    case 2: return launch_fwd_d64(p, dtype, st, ws);
    case 3: return launch_fwd_d96(p, dtype, st, ws);
    case 4: return launch_fwd_d128(p, dtype, st, ws);
    case 5: return launch_fwd_d160(p, dtype, st, ws);
    case 6: return launch_fwd_d192(p, dtype, st, ws);
    case 7: return launch_fwd_d224(p, dtype, st, ws);
    default: return launch_fwd_d256(p, dtype, st, ws);
  }
}

// Merge of the key-split partials: one thread per (row, 4 head dims). Row r belongs to work
// item w = r / br (query tile, head, sequence, decoded as the forward does) and is query
// qt*br + r % br of that sequence; rows past the sequence's end are left alone.
// LSE = m + log(sum_s exp(lse_s - m)), O = sum_s exp(lse_s - LSE) O_s; a row no split saw gets
// O = 0 and LSE = -inf, as in the unsplit kernel. Every share writes every row of its work
// item (a share without keys writes O = 0, LSE = -inf). All NMAX >= n shares' values are loaded
// before any is used (indices past n - 1 repeat the last share and are not summed), so the
// thread waits out one memory latency instead of one per share; the sum runs in share order.
template <typename T, int NMAX, class PGT>
__global__ __launch_bounds__(256) void fwd_split_combine_kernel(FableFwdParams p, FwdSplit sp, PGT pg) {
  constexpr bool PG = std::is_same<PGT, FwdPaged>::value;
  const int ch = p.HD / 4;
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= sp.rows * ch) return;
  const long long r = gid / ch;
  const int c = (int)(gid - r * ch);
  const int w = (int)(r / sp.br), qti = w % sp.nqt, zh = w / sp.nqt;
  const int gp = PG ? p.gqa : 1, nheads = p.NH / gp;
  const int z = zh / nheads;
  int h = (zh % nheads) * gp;
  const int qt = p.causal ? sp.nqt - 1 - qti : qti;
  int q = qt * sp.br + (int)(r - (long long)w * sp.br);
  long long orow, lrow;  // elements of this row in O and LSE
  if constexpr (PG) {    // packed rows: token q / gqa, head q % gqa of the group
    const PagedView v = paged_view(p, pg, z);
    if (q >= v.SQ * gp) return;
    const int t = q / gp;
    h += q - t * gp;
    orow = v.o0 + (long long)h * p.sO.h + (long long)t * p.sO.s;
    lrow = v.lse0 + (long long)h * p.lse_sh + (long long)t * pg.lse_sq;
  } else {
    const SeqView sv = seq_view(p, z, h);
    if (q >= sv.SQ) return;
    orow = sv.o0 + (long long)h * p.sO.h + (long long)q * p.sO.s;
    lrow = sv.lse0 + q;
  }
  float ls[NMAX];
  f32x4 ov[NMAX];
  // (paged instances: a share without keys writes its LSE only; many shares then load first the LSEs and O
  // where there is one)
  constexpr bool kTwo = PG && NMAX > 8;
#pragma unroll
  for (int k = 0; k < NMAX; k++) {
    const long long rk = (long long)min(k, sp.n - 1) * sp.rows + r;
    ls[k] = sp.lse[rk];
    if (!kTwo) ov[k] = *(const f32x4*)(sp.o + rk * p.HD + 4 * c);
  }
  if constexpr (kTwo) {
#pragma unroll
    for (int k = 0; k < NMAX; k++)
      if (k < sp.n && ls[k] != -INFINITY) ov[k] = *(const f32x4*)(sp.o + ((long long)k * sp.rows + r) * p.HD + 4 * c);
  }
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < NMAX; k++)
    if (k < sp.n) m = fmaxf(m, ls[k]);
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  float wsum = 0.0f;
  if (m != -INFINITY) {
#pragma unroll
    for (int k = 0; k < NMAX; k++) {
      if (k < sp.n) {
        const float wk = __expf(ls[k] - m);
        wsum += wk;
        if (!PG || ls[k] != -INFINITY) acc += wk * ov[k];
      }
    }
  }
  const float inv = m != -INFINITY ? 1.0f / wsum : 0.0f;
  typename Dt<T>::V4 o;
#pragma unroll
  for (int e = 0; e < 4; e++) o[e] = (T)(acc[e] * inv);
  *(u32x2*)((T*)p.O + orow + 4 * c) = __builtin_bit_cast(u32x2, o);
  if (c == 0 && p.LSE) p.LSE[lrow] = m != -INFINITY ? m + __logf(wsum) : -INFINITY;
}

template <typename T, class PGT>
static void launch_combine(const FableFwdParams& p, const FwdSplit& sp, PGT pg, dim3 grid, hipStream_t st) {
  if (sp.n <= 2)
    hipLaunchKernelGGL((fwd_split_combine_kernel<T, 2, PGT>), grid, dim3(256), 0, st, p, sp, pg);
  else if (sp.n <= 4)
    hipLaunchKernelGGL((fwd_split_combine_kernel<T, 4, PGT>), grid, dim3(256), 0, st, p, sp, pg);
  else if (sp.n <= 8)
    hipLaunchKernelGGL((fwd_split_combine_kernel<T, 8, PGT>), grid, dim3(256), 0, st, p, sp, pg);
  else if (sp.n <= 16)
    hipLaunchKernelGGL((fwd_split_combine_kernel<T, 16, PGT>), grid, dim3(256), 0, st, p, sp, pg);
  else if constexpr (std::is_same<PGT, FwdPaged>::value)
    hipLaunchKernelGGL((fwd_split_combine_kernel<T, 32, PGT>), grid, dim3(256), 0, st, p, sp, pg);
}

template <class PGT>
static int launch_combine_any(const FableFwdParams& p, const FwdSplit& sp, PGT pg, int nmax, int dtype, hipStream_t st) {
  if (sp.n < 2 || sp.n > nmax) return fail(FA_ERR_ARG, "fable_attn_fwd: %d key splits (2..%d)", sp.n, nmax);
  const long long items = sp.rows * (p.HD / 4);
  const dim3 grid((unsigned)((items + 255) / 256));
  if (dtype == FA_F16)
    launch_combine<_Float16>(p, sp, pg, grid, st);
  else
    launch_combine<__bf16>(p, sp, pg, grid, st);
  return launch_status("fable_attn_fwd (split merge)");
}
int launch_fwd_split_combine(const FableFwdParams& p, int dtype, const FwdSplit& sp, hipStream_t st) {
  return launch_combine_any(p, sp, NoPaged{}, 16, dtype, st);
}
int launch_fwd_split_combine_paged(const FableFwdParams& p, const FwdPaged& pg, int dtype, const FwdSplit& sp, hipStream_t st) {
  return launch_combine_any(p, sp, pg, 32, dtype, st);
}

// checks shared by the entry points (a workspace query needs no tensor pointers); 1 when the
// call has nothing to do
static int fwd_check(FableFwdParams& p, int dtype, bool query, int& rc) {
  rc = FA_OK;
  if (!query && (!p.Q || !p.K || !p.V || !p.O))
    return rc = fail(FA_ERR_ARG, "fable_attn_fwd: null tensor pointer"), 1;
  if (p.NH <= 0 || p.gqa <= 0 || p.NH % p.gqa) return rc = fail(FA_ERR_ARG, "fable_attn_fwd: NH=%d gqa=%d", p.NH, p.gqa), 1;
  if (!(p.dropout_p >= 0.0f && p.dropout_p < 1.0f)) return rc = fail(FA_ERR_ARG, "fable_attn_fwd: dropout_p=%g", p.dropout_p), 1;
  if ((p.cu_q == nullptr) != (p.cu_k == nullptr)) return rc = fail(FA_ERR_ARG, "fable_attn_fwd: cu_q and cu_k go together"), 1;
  if (!p.cu_q && p.batch <= 0) return 1;
  if (p.SQ < 0 || p.SK < 0) return rc = fail(FA_ERR_ARG, "fable_attn_fwd: SQ=%d SK=%d", p.SQ, p.SK), 1;
  // A window or chunk at least as long as the sequences bounds nothing; dropping it keeps every
  // mask bound the kernels form (row + delta + window) inside 32-bit range.
  if (p.win_left >= p.SK) p.win_left = -1;
  if (p.win_right >= p.SQ) p.win_right = -1;
  if (p.attn_chunk >= p.SK) p.attn_chunk = 0;
  if (dtype != FA_F16 && dtype != FA_BF16 && dtype != FA_F32)
    return rc = fail(FA_ERR_DTYPE, "fable_attn_fwd: dtype %d not implemented (fp16/bf16/fp32)", dtype), 1;
  return 0;
}

static int fwd_run(FableFwdParams p, int dtype, FwdWs& ws, hipStream_t st) {
  int rc;
  if (fwd_check(p, dtype, ws.query, rc)) return rc;
  if (dtype == FA_F32) return ws.query ? FA_OK : launch_fwd_f32(p, st);
  return dispatch_hd(p, dtype, st, ws);
}

}  // namespace fa

extern "C" int fable_attn_fwd(FableFwdParams p, int dtype, void* stream) {
  fa::FwdWs ws{nullptr, 0, false, 0};
  return fa::fwd_run(p, dtype, ws, (hipStream_t)stream);
}

extern "C" int64_t fable_attn_fwd_ws_bytes(FableFwdParams p, int dtype) {
  fa::FwdWs ws{nullptr, 0, true, 0};
  if (fa::fwd_run(p, dtype, ws, nullptr) != FA_OK) return -1;
  return ws.need;
}

extern "C" int fable_attn_fwd_ws(FableFwdParams p, int dtype, void* ws_ptr, int64_t ws_bytes, void* stream) {
  fa::FwdWs ws{ws_ptr, ws_bytes, false, 0};
  return fa::fwd_run(p, dtype, ws, (hipStream_t)stream);
}

// ------------------------------------------------------------------ packed prompts over a paged cache
namespace fa {

// whether the paged instances serve the call: fp16/bf16, no dropout, pages of at least 16 rows, a
// head dim whose kernel width is 64, 128 or 256 (the other widths would run with a third of their
// columns zero: for those a gather and the packed forward is the faster way), row strides of which 16
// rows stay within the 32-bit offsets of a load, pages under 2^31 elements apart, a table of fewer than
// 2^31 entries
static bool paged_served(const FableFwdParams& p, const FablePagedKV& kv, int dtype) {
  if (dtype != FA_F16 && dtype != FA_BF16) return false;
  if (p.HD <= 0 || p.HD > 256 || p.HD % 8 || p.dropout_p > 0.0f) return false;
  const int w = (p.HD + 31) / 32 * 32;
  constexpr long long kMaxRow = 0x7FFFFFFF / (16 * 2);   // elements
  if (p.sK.s < 0 || p.sK.s > kMaxRow || p.sV.s < 0 || p.sV.s > kMaxRow) return false;
  if ((long long)p.batch * kv.max_blocks > 0x7FFFFFFF) return false;
  if (kv.k_page_stride < 0 || kv.k_page_stride > 0x7FFFFFFF || kv.v_page_stride < 0 || kv.v_page_stride > 0x7FFFFFFF) return false;
  return (w == 64 || w == 128 || w == 256) && kv.page >= 16 && (kv.page & (kv.page - 1)) == 0;
}

static int paged_run(FableFwdParams p, FablePagedKV kv, int dtype, FwdWs& ws, hipStream_t st) {
  const long long room = (long long)kv.max_blocks * kv.page;
  if (!p.cu_q || !p.cu_k) return fail(FA_ERR_ARG, "fable_attn_fwd_paged: cu_q and cu_k are needed");
  if (!ws.query && !kv.block_table) return fail(FA_ERR_ARG, "fable_attn_fwd_paged: null block_table");
  if (kv.max_blocks < 0 || room > 0x7FFFFFFF) return fail(FA_ERR_ARG, "fable_attn_fwd_paged: max_blocks=%d page=%d", kv.max_blocks, kv.page);
  p.SK = (int)room;
  int rc;
  if (fwd_check(p, dtype, ws.query, rc)) return rc;
  if (!paged_served(p, kv, dtype)) return fail(FA_ERR_ARG, "fable_attn_fwd_paged: head_dim=%d page=%d dtype=%d is not served", p.HD, kv.page, dtype);
  const FwdPaged pg{kv.block_table, -1, kv.max_blocks, __builtin_ctz((unsigned)kv.page), kv.k_page_stride, kv.v_page_stride,
                    nullptr, 0, nullptr, nullptr, 1};
  return launch_fwd_paged(p, pg, dtype, false, st, ws);
}

}  // namespace fa

extern "C" int64_t fable_attn_fwd_paged_ws_bytes(FableFwdParams p, FablePagedKV kv, int dtype) {
  if (!fa::paged_served(p, kv, dtype)) return -2;
  fa::FwdWs ws{nullptr, 0, true, 0};
  if (fa::paged_run(p, kv, dtype, ws, nullptr) != FA_OK) return -1;
  return ws.need;
}

extern "C" int fable_attn_fwd_paged(FableFwdParams p, FablePagedKV kv, int dtype, void* ws_ptr, int64_t ws_bytes, void* stream) {
  fa::FwdWs ws{ws_ptr, ws_bytes, false, 0};
  return fa::paged_run(p, kv, dtype, ws, (hipStream_t)stream);
}
