// decode.hip — paged-KV split-KV decode for gfx950: KV append, partial attention per split,
// LSE-weighted combine.
//
// Replaces the reference decode (kernels/fa_decode.hip: fd_partial :57-252, fd_combine
// :255-272, fd_append :275-302, launcher :319-362) with the same FableDecParams contract
// (include/fable_attn_abi.h) and a different design:
//  * one workgroup (4 waves) per (kv head, group of 16 rows, run of a sequence's keys): the new
//    tokens x q heads that share a kv head are packed into the N=16 dimension of
//    v_mfma_f32_16x16x32, so K and V are read from HBM once per kv head whatever the GQA ratio and
//    for up to 16 rows of drafted tokens (4 tokens of 4 heads over 32000 keys: 66 -> 33 us, one
//    pass per token before); fp32: one workgroup per new token;
//  * K and V rows are read from the paged cache in whole rows (consecutive lanes cover one
//    row) and staged per wave in LDS; S^T = K . Q^T reads its A operand (16 bytes of one key
//    row per lane) back from the K slice, and the 16x16 result leaves every lane with one head
//    and four keys;
//  * P^T is the B operand of O^T = V^T . P^T (v_mfma_f32_16x16x16) without leaving registers;
//    V is read back from its slice transposed with ds_read_b64_tr_b16;
//  * each wave streams its own 16-key chunks (fp32: 32-key) with no barriers in the loop; the
//    four waves merge in LDS at the end and write one (max, sum, acc[HD]) partial per head and
//    split;
//  * the combine kernel merges the splits (natural-log LSE optional);
//  * appending new_k/new_v (with rotary on k) needs no synchronisation of the device (the
//    reference's hipDeviceSynchronize(), fa_decode.hip:348-351): one new token of a single sequence or
//    of a dense cache is written by the workgroups that read it, all others by a kernel earlier in
//    the same stream.
// Scores are handled in the log2 domain; partial maxima are stored in log2 units.
#include <mutex>
#include <type_traits>

#include "attn_device.hpp"
#include "fwd_common.hpp"
#include "status.hpp"

namespace fa {

static int dec_checked(FableDecParams p, int dtype, void* stream, const void* new_k, const void* new_v);

constexpr int kDecChunk = 32;  // keys per wave iteration of the fp32 kernel; splits are multiples
constexpr int kDecKeys = 16;   // keys per wave iteration of the fp16/bf16 kernel
constexpr int kDecWaves = 4;
static_assert(kDecKeys <= 16, "a chunk spans at most two pages of >= 16 rows (SPT)");

__device__ __forceinline__ float xor16_max(float x) {
  return fmaxf(x, __shfl_xor(x, 16));
}
__device__ __forceinline__ float xor16_sum(float x) { return x + __shfl_xor(x, 16); }

// Rows of a (sequence, K/V head): its nq new tokens x the gqa q heads of its group, token first;
// workgroups take them in groups of 16. The keys of a sequence some row sees are [lo, hi); row
// masks cut them down (a row of token tk sees [max(leftpad, pos - window + 1), ctx + (append ? tk +
// 1 : 0))). With `append` the span reaches down to ctx, so that it holds every new key.
struct DecSpan {
  int ctx, lo, hi;
};
// The lengths and tables are read as constant memory, which no kernel here writes: uniform entries
// then come by scalar loads (the kernels' own stores otherwise turn them into vector loads, whose
// in-order counter they would share with the row loads: C4 311 -> 319 us).
typedef const __attribute__((address_space(4))) int* cint_ptr;
__device__ __forceinline__ cint_ptr cmem(const int* p) { return (cint_ptr)(uintptr_t)p; }
__device__ __forceinline__ int dec_room(const FableDecParams& p) {
  return (int)min((long long)p.max_blocks * p.page, 0x7FFFFFFFLL);
}
__device__ __forceinline__ int dec_lo(const FableDecParams& p, int b, int ctx, int tk) {
  int lo = p.leftpad ? cmem(p.leftpad)[b] : 0;
  if (p.window >= 0) lo = max(lo, ctx + tk - p.window + 1);
  return max(lo, 0);
}
__device__ __forceinline__ int dec_hi(const FableDecParams& p, int ctx, int tk, int append) {
  return min(ctx + (append ? tk + 1 : 0), dec_room(p));
}
__device__ __forceinline__ DecSpan dec_span(const FableDecParams& p, int b, int append) {
  DecSpan r;
  r.ctx = cmem(p.ctx_len)[b];
  r.lo = dec_lo(p, b, r.ctx, 0);
  if (append) r.lo = max(min(r.lo, r.ctx), 0);
  r.hi = dec_hi(p, r.ctx, p.nq - 1, append);
  return r;
}

// How a call's keys are shared out when the caller sets no split count (p.nsplit 0). The lengths
// stay on the device, so every workgroup works out the shares by itself, from units of kUnit keys (a
// sequence has one at least):
//  * even: `parts` workgroups per (K/V head, row group); each sequence is cut into runs of `per`
//    units, `per` the least for which the runs fit the parts, so every workgroup has one run at
//    most. Taken where that is at most a quarter above an even share (few or alike sequences), or
//    kSegUnits units: a stream's workgroup pays a second segment, which costs about as much.
//  * stream: otherwise (many sequences of unequal lengths) the sequences' units follow one another
//    and each workgroup (two per part when there are more sequences than parts) takes as many, whatever sequences they belong to.
// A sequence that lies in one workgroup is finished there; of the others each writes a partial record
// (a stream's workgroup one for a sequence it goes on with, slot 0, and one for a sequence that goes
// on after it, slot 1). Two equal splits per sequence, the host's choice before, left 48 requests of 64
// to 8192 keys (Hq 64 / Hk 8, D 128) waiting for the longest: 142 us, 125 as a stream.
constexpr int kUnit = kDecKeys * kDecWaves;
__device__ __forceinline__ int dec_units(const DecSpan& r) { return max((r.hi - r.lo + kUnit - 1) / kUnit, 1); }
// inclusive prefix sum over the wave (row shifts within 16 lanes, then two broadcasts)
__device__ __forceinline__ int wave_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}
__device__ __forceinline__ int wave_sum(int x) { return __builtin_amdgcn_readlane(wave_scan(x), 63); }
// Every wave for itself: lane l holds the span of sequence base + l, read from memory once for
// batches of up to 64 sequences (a chain of dependent loads ahead of the first row load is what a
// short segment takes longest for).
struct DecShare {
  DecSpan mine;
  int units;        // of sequence base + lane; 0 past the batch
  int base;
  int total, per;   // units of the call, units per run (even) or workgroup (stream)
  bool even;
  __device__ __forceinline__ void load(const FableDecParams& p, int append, int b0, int lane) {
    base = b0;
    mine = DecSpan{0, 0, 0};
    units = 0;
    if (b0 + lane < p.batch) {
      mine = dec_span(p, b0 + lane, append);
      units = dec_units(mine);
    }
  }
  // sum over the batch of f(units); sequence 0's lanes are loaded afterwards
  template <typename F>
  __device__ __forceinline__ int sum(const FableDecParams& p, int append, int lane, F&& f) {
    int t = 0;
#pragma nounroll
    for (int b0 = (p.batch - 1) & ~63; b0 >= 0; b0 -= 64) {
      if (b0 != base) load(p, append, b0, lane);
      t += wave_sum(f(units));
    }
    return t;
  }
  __device__ __forceinline__ void init(const FableDecParams& p, int append, int parts, int lane) {
    load(p, append, 0, lane);
    total = sum(p, append, lane, [](int u) { return u; });
    const int least = max((int)((unsigned)(total + parts - 1) / (unsigned)parts), 1);
    even = false;
    if (p.batch <= parts) {
#pragma nounroll
      for (per = least; 4 * per <= 5 * least || per <= least + kSegUnits; per += max(per >> 4, 1)) {
        if (sum(p, append, lane, [=](int u) { return (int)((unsigned)(u + per - 1) / (unsigned)per); }) <= parts) {
          even = true;
          break;
        }
      }
    }
    if (!even) per = p.batch <= parts ? least : (least + 1) / 2;
  }
  // items: runs (even) or units (stream) of a sequence
  __device__ __forceinline__ int items(int u) const { return even ? (int)((unsigned)(u + per - 1) / (unsigned)per) : u; }
  __device__ __forceinline__ DecSpan span(int b) const {
    const int l = b - base;
    return DecSpan{__builtin_amdgcn_readlane(mine.ctx, l), __builtin_amdgcn_readlane(mine.lo, l), __builtin_amdgcn_readlane(mine.hi, l)};
  }
  // the sequence that holds item `at`, and its first item (p.batch: no such item); after init
  __device__ __forceinline__ int seek(const FableDecParams& p, int append, int at, int lane, int& first) {
    first = 0;
#pragma nounroll
    for (;;) {
      const int inc = wave_scan(items(units)), sum = __builtin_amdgcn_readlane(inc, 63);
      if (at >= first + sum) {
        first += sum;
        if (base + 64 >= p.batch) return p.batch;
        load(p, append, base + 64, lane);
        continue;
      }
      const int n = __popcll(__builtin_amdgcn_ballot_w64(first + inc <= at));   // sequences that end before `at`
      if (n > 0) first += __builtin_amdgcn_readlane(inc, n - 1);
      return base + n;
    }
  }
  // (at least 4 units per run and streams from a quarter above the even share on: 24 sequences of 500 keys, Hq 32 /
  // Hk 8, D 128, 21.3 us, 19.0 now; 3 of 500 13.7 and 11.6; 5 of 300 14.1 and 11.2)
  static constexpr int kSegUnits = 6;
};

// floats ahead of the records: two ints per sequence, for the combine
__host__ __device__ inline long long dec_meta_floats(const FableDecParams& p) { return (2ll * p.batch + 63) / 64 * 64; }

// The partial kernel's argument. The phases that only some workgroups run (the shares, the append)
// read it again from the kernel argument segment: the phases together use most of the 40 fields,
// and held for the whole kernel they spilled some 80 scalar registers.
struct DecArgs : FableDecParams {
  const void *nk, *nv;                  // the new key and value of each sequence, or null
  // block table: entry i of sequence b is table[b * max_blocks + i] (tmask -1), or b * max_blocks + i
  // for a dense cache without one (tmask 0: table is any readable address, its value masked off; no
  // branch, which would wait for the load at once)
  const int* table;
  int tmask;
  int page_shift, ngrp, flags, parts, nkv;
};
__device__ __forceinline__ DecArgs dec_reload() {
  auto k = (const __attribute__((address_space(4))) uint64_t*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  struct {
    uint64_t w[sizeof(DecArgs) / 8];
  } raw;
  static_assert(sizeof(raw) == sizeof(DecArgs), "whole words");
#pragma unroll
  for (int i = 0; i < (int)(sizeof(DecArgs) / 8); i++) raw.w[i] = k[i];
  return __builtin_bit_cast(DecArgs, raw);
}

// SPT (page >= 16): the block-table entries of a chunk are fetched by scalar loads. A chunk of
// 16 keys touches at most two pages then, and each lane selects its row's entry from the two.
// Per-lane table loads share the in-order vector-memory counter with the row loads, so a wave
// waiting for its next entries also waited for the rows issued before them (the chunk in
// flight): C4 +1% with the scalar loads (+4% in a read probe). Smaller pages (a dense cache of
// fewer than 16 rows) keep per-lane loads.
// flags: bit 0 new keys were appended (kDecAppend), bit 1 the kernel writes the final output and
// LSE itself (kDecFinal: one split, no combine launch)
constexpr int kDecAppend = 1, kDecFinal = 2;
template <typename T, int HD, bool FEAT, bool SPT, bool SHARE>
__global__ __launch_bounds__(256) void dec_partial_kernel(DecArgs p) {
  const int append = p.flags & kDecAppend, page_shift = p.page_shift;
  using V8 = typename Dt<T>::V8;
  constexpr int NDS = HD / 32;  // S^T contraction steps
  constexpr int NDB = HD / 16;  // 16-row blocks of O^T
  constexpr int RCH = HD / 8;   // 16-byte chunks per key row
  static_assert(RCH >= 8, "swizzle needs >= 8 chunks per row");
  // one LDS region, reused: q staging (fp32) before the loop, per-wave V chunks in the loop,
  // the four waves' accumulators after it; per-wave K chunks in a region of their own
  __shared__ __attribute__((aligned(16))) char vraw[kDecWaves * 16 * HD * 4];
  __shared__ __attribute__((aligned(16))) char kraw[kDecWaves * kDecKeys * HD * 2];
  __shared__ float red_m[kDecWaves][16], red_l[kDecWaves][16];
  static_assert(16 * HD * 4 <= sizeof(vraw), "q staging fits the V region");
  static_assert(kDecWaves * kDecKeys * HD * 2 <= sizeof(vraw), "the V slices fit the V region");
  float (*qsh)[HD] = (float (*)[HD])vraw;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lg = lane >> 4, lh = lane & 15;  // lane group (0..3), lane in group
  // (kv head, row group) fastest: the workgroups reading the interleaved heads of the same cache
  // pages are dispatched together, the row groups of one head to the same XCD where the heads
  // are a multiple of 8
  // (scalar divisions stand in a chain of some hundred cycles each ahead of the first load: the grid's
  // axes and the host's K/V head count leave none for calls of up to 16 rows)
  const int NKV = p.nkv, HDr = p.HD, nq = p.nq, gqa = p.gqa, NH = p.NH;
  const int X = gridDim.x, hgl = blockIdx.x, grp = p.ngrp > 1 ? hgl / NKV : 0, kvh = hgl - grp * NKV;
  const int r0 = 16 * grp, hg = min(16, nq * gqa - r0);  // rows of this group
  // row g: token, q head and index in q, o and lse
  auto row_tok = [&](int g) {
    int t = 0;
    if (nq > 1) t = (int)((unsigned)(r0 + g) / (unsigned)gqa);   // (a division per row: not for one token)
    return t;
  };
  auto row_of = [&](int b, int g) {
    const int tok = row_tok(g);
    return (long long)(b * nq + tok) * NH + kvh * gqa + (r0 + g - tok * gqa);
  };
  auto args = [&]() -> DecArgs {   // (the fixed grid's instances hold them)
    if constexpr (SHARE) return dec_reload();
    return p;
  };
  // segments: a stream part's (sequence, run of keys), or the one split of the grid
  DecShare str;
  int at = 0, at_end = 0, sq = 0, first = 0;  // (units; sq: the sequence that holds `at`, first: its first)
  if constexpr (SHARE) {
    const DecArgs p = dec_reload();
    str.init(p, append, p.parts, lane);
    const int part = blockIdx.y;
    if (str.even) {
      sq = str.seek(p, append, part, lane, first);
      if (sq >= p.batch) return;
      at = (part - first) * str.per;   // (this sequence's units from 0 on)
      at_end = at + str.per;
      first = 0;
    } else {
      at = part * str.per;
      at_end = min(at + str.per, str.total);
      if (at >= at_end) return;
      sq = str.seek(p, append, at, lane, first);
    }
  }
  for (bool more = true; more;) {
  const int b = SHARE ? sq : (int)blockIdx.y;
  // q rows of this group, loaded while the lengths are on their way: one 16-byte load per thread and
  // chunk, row index clamped (rows past the group are zeroed after the load)
  constexpr int NQI = (16 * RCH + 255) / 256;
  u32x4 qraw[NQI];
  {
    const DecArgs p = args();
#pragma unroll
    for (int u = 0; u < NQI; u++) {
      const int i = min(tid + 256 * u, 16 * RCH - 1), g = i / RCH, c = i % RCH;
      qraw[u] = *(const u32x4*)((const T*)p.q + row_of(b, min(g, hg - 1)) * HDr + (8 * c < HDr ? 8 * c : 0));
    }
  }
  DecSpan sp;
  if constexpr (!SHARE) sp = dec_span(p, b, append);
  int start, end;
  float* rec = nullptr;  // record of row 0 (rows rec_step apart); null: the final output
  long long rec_step = HDr + 2;
  if constexpr (SHARE) {
    const DecArgs p = dec_reload();
    if (b >= str.base + 64) str.load(p, append, b, lane);
    sp = str.span(b);
    const int units = dec_units(sp), stop = min(at_end, first + units);
    start = sp.lo + (at - first) * kUnit;
    end = min(sp.lo + (stop - first) * kUnit, sp.hi);
    const bool begins = at == first;
    const int part = blockIdx.y;
    // where the combine finds this sequence's records: the first one's index, and their count
    // (negative for a stream, whose later ones are in slot 0)
    if (begins && hgl == 0 && tid == 0) {
      const int n = str.even ? str.items(units) : (int)((unsigned)(first + units - 1) / (unsigned)str.per) - part + 1;
      ((int*)p.scratch)[2 * b] = 2 * part + (str.even ? 0 : 1);
      ((int*)p.scratch)[2 * b + 1] = str.even ? n : -n;
    }
    if (!(begins && stop == first + units))
      rec = p.scratch + dec_meta_floats(p) + ((2ll * part + (begins && !str.even ? 1 : 0)) * X + hgl) * 16 * (HDr + 2);
    at = stop;
    first += units;
    sq++;
    more = !str.even && at < at_end;
  } else {
    const int n = max(sp.hi - sp.lo, 0);
    const int share = p.nsplit > 1 ? (int)((unsigned)(n + p.nsplit - 1) / (unsigned)p.nsplit) : n;
    const int chunk = (share + kDecChunk - 1) / kDecChunk * kDecChunk;
    start = sp.lo + (int)blockIdx.z * chunk;
    end = min(start + chunk, sp.hi);
    if (!(p.flags & kDecFinal)) {
      rec = p.scratch + (long long)blockIdx.z * (HDr + 2);
      rec_step = (long long)p.nsplit * (HDr + 2);   // rows are indexed as in q
    }
    more = false;
  }
  const int ctx = sp.ctx;
  start = __builtin_amdgcn_readfirstlane(start);
  end = __builtin_amdgcn_readfirstlane(end);

  // ---- a single new key (nk) -> the cache (rotated k, v), by the workgroups that read it next: an
  // append kernel of its own cost 3 us ahead of a 9 us decode. (Row groups of one head write the
  // same bytes. Which calls come here: dec_fuses_append. Several tokens keep the kernel: written here
  // one after another they cost more.)
  if (append && ctx >= start && ctx < end) {
    const DecArgs p = dec_reload();
    if (p.nk) {
      const int j = ctx >> page_shift, rdim = p.rotary ? (p.rotary_dim > 0 ? p.rotary_dim : HDr) : 0, half = rdim / 2;
      const int blk = p.block_table ? p.block_table[(long long)b * p.max_blocks + j] : b * p.max_blocks + j;
      const long long dst = (((long long)blk * p.page + (ctx & (p.page - 1))) * NKV + kvh) * HDr, src = ((long long)b * NKV + kvh) * HDr;
      T* kd = (T*)p.Kc + dst;
      const int vc = 8 * (tid - 224);   // (at most 128 pairs of k; the last 32 threads carry v)
      if (vc >= 0 && vc < HDr) *(u32x4*)((T*)p.Vc + dst + vc) = *(const u32x4*)((const T*)p.nv + src + vc);
      if (tid >= rdim && tid < HDr) kd[tid] = ((const T*)p.nk)[src + tid];
      if (tid < half) {
        const long long at = (long long)(p.rotary_pos ? p.rotary_pos[b] : ctx) * half + tid;
        const float c = p.cos[at], sn = p.sin[at];
        const int ia = p.rotary == 1 ? tid : 2 * tid, ib = p.rotary == 1 ? tid + half : 2 * tid + 1;
        const float x = (float)((const T*)p.nk)[src + ia], y = (float)((const T*)p.nk)[src + ib];
        kd[ia] = (T)(x * c - y * sn);
        kd[ib] = (T)(y * c + x * sn);
      }
      __syncthreads();  // in the cache (this CU's view of it) before the rows are read below
    }
  }

  // ---- q rows of this group -> LDS (fp32)
  // A head dim HDr = p.HD below the kernel width HD (a multiple of 8) runs with zero columns
  // HDr..HD-1 in q, K and V (rows in memory are HDr long); only HDr output columns are kept.
  bool qsplit;
  {
  const DecArgs p = args();
  qsplit = p.rotary != 0;
#pragma unroll
  for (int u = 0; u < NQI; u++) {
    const int i = tid + 256 * u, g = i / RCH, c = i % RCH;
    const bool cok = 8 * c < HDr;
    const V8 v = bitcast<V8>(qraw[u]);
    if (i < 16 * RCH)
#pragma unroll
      for (int e = 0; e < 8; e++) qsh[g][8 * c + e] = g < hg && cok ? (float)v[e] : 0.0f;
  }
  __syncthreads();
  if (p.rotary) {
    const int rdim = p.rotary_dim > 0 ? p.rotary_dim : HDr, half = rdim / 2;
    const int rbase = p.rotary_pos ? p.rotary_pos[b] : ctx;
    for (int i = tid; i < hg * half; i += 256) {
      const int g = i / half, j = i % half, rp = rbase + row_tok(g);
      const float c = p.cos[(long long)rp * half + j], s = p.sin[(long long)rp * half + j];
      const int ia = p.rotary == 1 ? j : 2 * j, ib = p.rotary == 1 ? j + half : 2 * j + 1;
      const float x = qsh[g][ia], y = qsh[g][ib];
      qsh[g][ia] = x * c - y * s;
      qsh[g][ib] = y * c + x * s;
    }
    __syncthreads();
  }
  }
  // Q^T as the B operand: lane holds head lh, head-dim 32*ds + 8*lg + e. A rotated q is not
  // representable in T; it is carried as hi + lo (two MFMAs per step) so rotation costs no
  // precision beyond fp32.
  V8 qb[NDS], ql[NDS];
#pragma unroll
  for (int ds = 0; ds < NDS; ds++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float x = qsh[lh][32 * ds + 8 * lg + e];
      const T hi = (T)x;
      qb[ds][e] = hi;
      ql[ds][e] = (T)(x - (float)hi);
    }
  __syncthreads();  // q staging is dead from here on: the region becomes the V chunk buffers

  f32x4 oacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; db++) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.0f;
  const float c_log2 = p.scale * kLog2e;
  const int tok = row_tok(min(lh, hg - 1)), qpos = ctx + tok;  // this lane's row (lh)
  const int rlo = max(dec_lo(p, b, ctx, tok), start), rspan = max(min(dec_hi(p, ctx, tok, append), end) - rlo, 0);
  const float slope = (FEAT && p.alibi && lh < hg) ? p.alibi[kvh * p.gqa + (r0 + lh - tok * p.gqa)] : 0.0f;
  const T* Kc = (const T*)p.Kc;
  const T* Vc = (const T*)p.Vc;
  const cint_ptr bt = cmem(p.table) + (long long)b * (p.max_blocks & p.tmask);
  const int blk0 = b * p.max_blocks, tmask = p.tmask;
  auto entry = [&](int raw, int i) { return (raw & tmask) | ((blk0 + i) & ~tmask); };
  const int pmask = p.page - 1;
  T* vb = (T*)vraw + wave * kDecKeys * HD;
  T* kbuf = (T*)kraw + wave * kDecKeys * HD;

  // Keys of a chunk are clamped into [start, end-1] (masked in the softmax), so every load is
  // unconditional. Block-table entries are fetched ahead of the row loads that use them, so the
  // K/V row loads of a chunk issue back to back instead of behind their table lookups.
  constexpr int NVI = kDecKeys * RCH / 64;  // K (and V) row loads per lane per chunk
  const int last = end - 1;
  auto vkey = [&](int kc0, int i) { return min(kc0 + (64 * i + lane) / RCH, last); };
  // (entries are kept as read, and made pages where the rows are loaded: any use of one here would wait
  // for it, chunk by chunk; sidx: indices of sblk)
  int vblk[SPT ? 1 : NVI], sblk[2], sidx[2];
  auto table = [&](int kc0) {
    if constexpr (SPT) {
      const int b0 = kc0 >> page_shift, bl = last >> page_shift;  // wave-uniform
#pragma unroll
      for (int j = 0; j < 2; j++) {
        sidx[j] = min(b0 + j, bl);
        sblk[j] = bt[sidx[j] & tmask];
      }
    } else {
#pragma unroll
      for (int i = 0; i < NVI; i++) vblk[i] = bt[(vkey(kc0, i) >> page_shift) & tmask];
    }
  };
  // entry of load i's row: page (key >> page_shift) - (kc0 >> page_shift) of the chunk's two
  // (a key clamped to `last` lies in the chunk's last page, whose index the table clamped too)
  auto blk_of = [&](int kc0, int i, const int (&pg)[2]) {
    if constexpr (SPT) {
      const int j = (vkey(kc0, i) >> page_shift) - (kc0 >> page_shift);
      return j <= 0 ? pg[0] : pg[1];
    } else {
      return entry(vblk[i], vkey(kc0, i) >> page_shift);
    }
  };
  auto row_off = [&](int blk, int key) -> long long {
    return (((long long)blk * p.page + (key & pmask)) * NKV + kvh) * HDr;
  };
  // 16-byte chunks in the zero columns load the row's first chunk and are replaced by zeros
  const bool padded = HDr < HD;
  bool vok[NVI];
#pragma unroll
  for (int i = 0; i < NVI; i++) vok[i] = 8 * ((64 * i + lane) % RCH) < HDr;
  // K/V rows of the chunk at kc0: load i covers row (64i + lane) / RCH, 16-byte chunk
  // (64i + lane) % RCH of both caches, so consecutive lanes read whole rows. Loading K straight
  // into the MFMA A layout instead (16 keys x 64 bytes per load) read the cache ~12% slower.
  // The cache rows are read once per step: non-temporal loads keep them from displacing the
  // block table and q in the caches (C4: 368.6 -> 360.3 us for the partial kernel).
  auto load = [&](int kc0, u32x4 (&kr)[NVI], u32x4 (&vr)[NVI]) {
    int pg[2] = {0, 0};   // (formed on the scalar unit: after the selection it took 18 VALU per chunk)
    if constexpr (SPT) {
#pragma unroll
      for (int j = 0; j < 2; j++) pg[j] = __builtin_amdgcn_readfirstlane(entry(sblk[j], sidx[j]));
    }
#pragma unroll
    for (int i = 0; i < NVI; i++) {
      const int ch = (64 * i + lane) % RCH;
      const long long off = row_off(blk_of(kc0, i, pg), vkey(kc0, i)) + (vok[i] ? 8 * ch : 0);
      kr[i] = __builtin_nontemporal_load((const u32x4*)(Kc + off));
      vr[i] = __builtin_nontemporal_load((const u32x4*)(Vc + off));
    }
  };
  // zero columns of a padded head dim, put in where the rows are used (which waits for the
  // loads anyway; a select right after the loads would make the compiler wait there)
  auto zero_pad = [&](u32x4 (&kr)[NVI], u32x4 (&vr)[NVI]) {
    if (padded) {
#pragma unroll
      for (int i = 0; i < NVI; i++) {
        kr[i] = vok[i] ? kr[i] : u32x4{0, 0, 0, 0};
        vr[i] = vok[i] ? vr[i] : u32x4{0, 0, 0, 0};
      }
    }
  };
  // K slice: row r holds logical 16-byte chunk c at physical chunk c ^ kswz(r). The rows of
  // one 256-byte bank line share a pattern and consecutive lines differ, so the 16 lanes of an
  // A-operand read (16 rows, one chunk) and of a row write hit 16 different bank groups.
  // (A width whose chunk count is not a power of two XORs within aligned groups of the largest
  // power of two that divides it, so a chunk never leaves its row: 12 chunks at width 96 swizzle
  // in groups of 4.)
  constexpr int kRowsPerLine = HD >= 128 ? 1 : 128 / HD;
  constexpr int kSwzGroup = (RCH & -RCH) < 16 ? (RCH & -RCH) : 16;
  constexpr int kSwzMask = kSwzGroup - 1;
  auto kswz = [](int r) { return (r / kRowsPerLine) & kSwzMask; };
  // V slice: chunk c of row r at c ^ vswz(r), pairs of chunks for the transposing reads
  auto vswz = [](int r) { return kSwzGroup >= 8 ? 2 * (r & 3) : 2 * (r & 1); };
  // Each wave walks 16-key chunks with one register set: a chunk's rows go to LDS, the next
  // chunk's loads are issued, and the chunk is computed from LDS meanwhile. Table entries run
  // one chunk ahead. Keys past the end clamp to the last one. Read probes over the C4 cache
  // streamed fastest with about 8 KiB of rows in flight per wave (16 keys of K and V at
  // D=128); 32-key chunks with a second register set in flight read ~6% slower there.
  constexpr int kStep = kDecKeys * kDecWaves;
  const int kfirst = start + kDecKeys * wave;
  u32x4 kreg[NVI], vreg[NVI];
  if (kfirst < end) {
    table(kfirst);
    load(kfirst, kreg, vreg);
    table(kfirst + kStep);
  }
  for (int kc0 = kfirst; kc0 < end; kc0 += kStep) {
    zero_pad(kreg, vreg);
    // K and V -> this wave's LDS slices; the slices are the wave's own, and LDS operations of
    // one wave complete in order, so no barrier orders these writes against the reads below or
    // against the previous chunk's reads
#pragma unroll
    for (int i = 0; i < NVI; i++) {
      const int row = (64 * i + lane) / RCH, ch = (64 * i + lane) % RCH;
      *(u32x4*)(kbuf + row * HD + 8 * (ch ^ kswz(row))) = kreg[i];
      *(u32x4*)(vb + row * HD + 8 * (ch ^ vswz(row))) = vreg[i];
    }
    // the next chunk's rows are in flight during this chunk's products
    if (kc0 + kStep < end) {
      load(kc0 + kStep, kreg, vreg);
      table(kc0 + 2 * kStep);
    }
    // S^T = K . Q^T, A operand: lane (lg, lh) reads key row lh, head-dim chunk 4*ds + lg
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
    {
      V8 ka[NDS];
#pragma unroll
      for (int ds = 0; ds < NDS; ds++) ka[ds] = bitcast<V8>(*(const u32x4*)(kbuf + lh * HD + 8 * ((4 * ds + lg) ^ kswz(lh))));
#pragma unroll
      for (int ds = 0; ds < NDS; ds++) s = Dt<T>::mma16(ka[ds], qb[ds], s);
      if (qsplit) {
#pragma unroll
        for (int ds = 0; ds < NDS; ds++) s = Dt<T>::mma16(ka[ds], ql[ds], s);
      }
    }
    // logits (log2 domain) and masking: s[r] is key kc0 + 4*lg + r, head lh
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int key = kc0 + 4 * lg + r;
      float t;
      if (FEAT) {
        float x = s[r] * p.scale;
        if (p.softcap > 0.0f) x = p.softcap * tanh_exp(x / p.softcap);
        x += slope * (float)(key - qpos);
        t = x * kLog2e;
      } else {
        t = s[r] * c_log2;
      }
      t = (unsigned)(key - rlo) < (unsigned)rspan ? t : -INFINITY;
      s[r] = t;
      mx = fmaxf(mx, t);
    }
    mx = half_max(xor16_max(mx));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    const float corr = exp2_fast(m_run - m_use);
    float rs = 0.0f;
    typename Dt<T>::V4 pb;  // P^T, the B operand of the k=16 product: keys 4*lg + r, head lh
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float e = exp2_fast(s[r] - m_use);
      rs += e;
      pb[r] = (T)e;
    }
    l_run = l_run * corr + rs;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < NDB; db++) oacc[db] *= corr;
    // O^T += V^T . P^T, A operand by transposing LDS reads: lane lh of group lg addresses row
    // 4*lg + lh/4, head-dim 16*db + 4*(lh%4); it receives V[4*lg + r][16*db + lh]
#pragma unroll
    for (int db = 0; db < NDB; db++) {
      const int row = 4 * lg + (lh >> 2);
      const int col = 16 * db + 4 * (lh & 3);
      const int off = row * HD + 8 * ((col >> 3) ^ vswz(row)) + (col & 7);
      typedef short s4 __attribute__((ext_vector_type(4)));
      const s4 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s4*)((__attribute__((address_space(3))) T*)vb + off));
      oacc[db] = Dt<T>::mma16k16(bitcast<typename Dt<T>::V4>(t), pb, oacc[db]);
    }
  }

  // ---- merge the four waves: per head max, sum and O^T accumulators through LDS
  const float l_grp = half_sum(xor16_sum(l_run));
  __syncthreads();  // every wave is done with its V slice: reuse it for the accumulators
  float* red_o = (float*)vraw;  // [wave][16 heads][HD]
  if (lg == 0) {
    red_m[wave][lh] = m_run;
    red_l[wave][lh] = l_grp;
  }
#pragma unroll
  for (int db = 0; db < NDB; db++)
#pragma unroll
    for (int r = 0; r < 4; r++) red_o[(wave * 16 + lh) * HD + 16 * db + 4 * lg + r] = oacc[db][r];
  __syncthreads();
  const DecArgs pe = args();
  for (int i = tid; i < hg * HDr; i += 256) {
    const int g = i / HDr, d = i % HDr;
    float gm = -INFINITY;
#pragma unroll
    for (int w = 0; w < kDecWaves; w++) gm = fmaxf(gm, red_m[w][g]);
    float l = 0.0f, acc = 0.0f;
    if (gm != -INFINITY) {
#pragma unroll
      for (int w = 0; w < kDecWaves; w++) {
        const float f = exp2_fast(red_m[w][g] - gm);
        l += f * red_l[w][g];
        acc += f * red_o[(w * 16 + g) * HD + d];
      }
    }
    const long long row = row_of(b, g);
    if (!rec) {
      // what the combine kernel computes from one split (its weight exp2(0) is exactly 1)
      const bool ok = gm != -INFINITY && l > 0.0f;
      ((T*)pe.o)[row * HDr + d] = (T)(ok ? acc / l : 0.0f);
      if (pe.lse_out && d == 0) pe.lse_out[row] = ok ? gm * kLn2 + __logf(l) : -INFINITY;
      continue;
    }
    float* out = rec + (SHARE ? g : row) * rec_step;
    if (d == 0) {
      out[0] = gm;
      out[1] = l;
    }
    out[2 + d] = acc;
  }
  if (more) __syncthreads();  // the merge has read the LDS regions before the next segment fills them
  }
}

// fp32 caches (the reference's decode serves fp16/bf16/fp32, fa_decode.hip:4,360): the same
// workgroup and wave split, on v_mfma_f32_16x16x4_f32. Lane (head lh, group lg) holds q dims
// lg*HD/4 + t as the B operand of S^T = K . Q^T, whose A operand is loaded straight from the
// paged cache (16 bytes of one key row per lane); P^T is the B operand of O^T = V^T . P^T,
// whose A operand is one float per lane (V[key 16kb + 4lg + j][16db + lh]), read from the cache
// as well (four 64-byte row segments per load). Rotation of q stays exact in fp32. Kernel
// widths HD = 64, 128, 256 serve every head dim p.HD that is a multiple of 8: rows are p.HD
// floats apart and the partial record holds the p.HD real columns. Columns past p.HD are read
// at a clamped column of the same row (always in bounds, no branch): for K the product meets
// q columns that are zero there, and for V it only fills O^T rows past p.HD, which are never
// stored. (Per-load branches here raised the kernel's scalar registers past the file and the
// 256-wide alibi variant then computed wrong logits; the clamped form keeps the register use
// of the full-width kernel.)
template <int HD, bool FEAT>
__global__ __launch_bounds__(256) void dec_partial_f32_kernel(FableDecParams p, int page_shift, int ngrp, int append) {
  constexpr int NQ = HD / 4;    // S^T contraction steps (q floats per lane)
  constexpr int NDB = HD / 16;  // 16-row blocks of O^T
  constexpr int QSTR = HD + 4;
  constexpr int QBYTES = 16 * QSTR * 4, OBYTES = kDecWaves * 16 * HD * 4;
  __shared__ __attribute__((aligned(16))) char raw[QBYTES > OBYTES ? QBYTES : OBYTES];
  __shared__ float red_m[kDecWaves][16], red_l[kDecWaves][16];
  float (*qsh)[QSTR] = (float (*)[QSTR])raw;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lg = lane >> 4, lh = lane & 15;
  const int b = blockIdx.y / p.nq, tk = blockIdx.y % p.nq;
  const int kvh = blockIdx.x / ngrp, hgi = blockIdx.x % ngrp;
  const int h0 = kvh * p.gqa + 16 * hgi, hg = min(16, p.gqa - 16 * hgi);
  const int sp = blockIdx.z;
  const int NKV = p.NH / p.gqa, HDr = p.HD;
  struct {
    int qpos, start, end;
  } rg;
  {
    const int ctx = p.ctx_len[b], lo = dec_lo(p, b, ctx, tk), hi = dec_hi(p, ctx, tk, append), n = max(hi - lo, 0);
    const int chunk = (((n + p.nsplit - 1) / p.nsplit) + kDecChunk - 1) / kDecChunk * kDecChunk;
    rg.qpos = ctx + tk;
    rg.start = lo + sp * chunk;
    rg.end = min(rg.start + chunk, hi);
  }

  const float* qg = (const float*)p.q + ((long long)(b * p.nq + tk) * p.NH + h0) * HDr;
  for (int i = tid; i < 16 * NQ; i += 256) {
    const int g = i / NQ, c = i % NQ;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    if (g < hg && 4 * c < HDr) v = *(const f32x4*)(qg + (long long)g * HDr + 4 * c);
#pragma unroll
    for (int e = 0; e < 4; e++) qsh[g][4 * c + e] = v[e];
  }
  __syncthreads();
  if (p.rotary) {
    const int rdim = p.rotary_dim > 0 ? p.rotary_dim : HDr, half = rdim / 2;
    const int rp = (p.rotary_pos ? p.rotary_pos[b] : p.ctx_len[b]) + tk;
    for (int i = tid; i < hg * half; i += 256) {
      const int g = i / half, j = i % half;
      const float c = p.cos[(long long)rp * half + j], s = p.sin[(long long)rp * half + j];
      const int ia = p.rotary == 1 ? j : 2 * j, ib = p.rotary == 1 ? j + half : 2 * j + 1;
      const float x = qsh[g][ia], y = qsh[g][ib];
      qsh[g][ia] = x * c - y * s;
      qsh[g][ib] = y * c + x * s;
    }
    __syncthreads();
  }
  float qreg[NQ];
#pragma unroll
  for (int t = 0; t < NQ; t++) qreg[t] = qsh[lh][lg * NQ + t];

  f32x4 oacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; db++) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.0f;
  const float c_log2 = p.scale * kLog2e;
  const float slope = (FEAT && p.alibi && lh < hg) ? p.alibi[h0 + lh] : 0.0f;
  const float inv_cap = p.softcap > 0.0f ? 1.0f / p.softcap : 0.0f;
  const float* Kc = (const float*)p.Kc;
  const float* Vc = (const float*)p.Vc;
  const int* bt = p.block_table + (long long)b * p.max_blocks;
  const int pmask = p.page - 1;
  const int last = rg.end - 1;
  auto row_off = [&](int key) -> long long {
    return (((long long)bt[key >> page_shift] * p.page + (key & pmask)) * NKV + kvh) * HDr;
  };
  constexpr int kStep = kDecChunk * kDecWaves;
  for (int kc0 = rg.start + kDecChunk * wave; kc0 < rg.end; kc0 += kStep) {
    // keys past the end clamp to the last one (masked below), so every load is unconditional
    f32x4 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; kb++) {
      const float* kr = Kc + row_off(min(kc0 + 16 * kb + lh, last));
      s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NQ / 4; u++) {
        const f32x4 a = *(const f32x4*)(kr + min(lg * NQ + 4 * u, HDr - 4));
#pragma unroll
        for (int e = 0; e < 4; e++) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], qreg[4 * u + e], s[kb], 0, 0, 0);
      }
    }
    // s[kb][r] is key kc0 + 16*kb + 4*lg + r, head lh
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int key = kc0 + 16 * kb + 4 * lg + r;
        float t;
        if (FEAT) {
          float x = s[kb][r] * p.scale;
          if (p.softcap > 0.0f) x = p.softcap * tanhf(x * inv_cap);
          x += slope * (float)(key - rg.qpos);
          t = x * kLog2e;
        } else {
          t = s[kb][r] * c_log2;
        }
        t = key < rg.end ? t : -INFINITY;
        s[kb][r] = t;
        mx = fmaxf(mx, t);
      }
    mx = half_max(xor16_max(mx));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    const float corr = exp2_fast(m_run - m_use);
    float rs = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float e = exp2_fast(s[kb][r] - m_use);
        rs += e;
        s[kb][r] = e;
      }
    l_run = l_run * corr + rs;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < NDB; db++) oacc[db] *= corr;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float* vr = Vc + row_off(min(kc0 + 16 * kb + 4 * lg + r, last));
#pragma unroll
        for (int db = 0; db < NDB; db++)
          oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[min(16 * db + lh, HDr - 1)], s[kb][r], oacc[db], 0, 0, 0);
      }
  }

  // ---- merge the four waves (as the fp16/bf16 kernel)
  const float l_grp = half_sum(xor16_sum(l_run));
  __syncthreads();  // q staging is dead: the region holds the accumulators
  float* red_o = (float*)raw;  // [wave][16 heads][HD]
  if (lg == 0) {
    red_m[wave][lh] = m_run;
    red_l[wave][lh] = l_grp;
  }
#pragma unroll
  for (int db = 0; db < NDB; db++)
#pragma unroll
    for (int r = 0; r < 4; r++) red_o[(wave * 16 + lh) * HD + 16 * db + 4 * lg + r] = oacc[db][r];
  __syncthreads();
  for (int i = tid; i < hg * HDr; i += 256) {
    const int g = i / HDr, d = i % HDr;
    float gm = -INFINITY;
#pragma unroll
    for (int w = 0; w < kDecWaves; w++) gm = fmaxf(gm, red_m[w][g]);
    float l = 0.0f, acc = 0.0f;
    if (gm != -INFINITY) {
#pragma unroll
      for (int w = 0; w < kDecWaves; w++) {
        const float f = exp2_fast(red_m[w][g] - gm);
        l += f * red_l[w][g];
        acc += f * red_o[(w * 16 + g) * HD + d];
      }
    }
    float* out = p.scratch + (((long long)(b * p.nq + tk) * p.NH + h0 + g) * p.nsplit + sp) * (HDr + 2);
    if (d == 0) {
      out[0] = gm;
      out[1] = l;
    }
    out[2 + d] = acc;
  }
}

// merge nsplit partials of one (token, head): grid (batch*nq, NH), block HD
template <typename T, int HD, int NC, bool STREAM = false>
__global__ __launch_bounds__(256) void dec_combine_kernel(FableDecParams p, int ngrp) {
  // one thread per column of the kernel width HD; the head dim p.HD <= HD sets the strides
  const int row = blockIdx.x, h = blockIdx.y, d = threadIdx.x, HDr = p.HD;
  const int dc = min(d, HDr - 1);  // threads past the head dim read a valid column, store nothing
  const float* base = p.scratch + ((long long)row * p.NH + h) * p.nsplit * (HDr + 2);
  // STREAM: the records of this row's sequence, one per part its units lie in; one part alone has
  // written the output already
  int ns = p.nsplit;
  long long rest = 0, step = HDr + 2;  // record s > 0 is at base + rest + s * step
  if constexpr (STREAM) {
    const int b = row / p.nq, tk = row - b * p.nq, slot0 = ((const int*)p.scratch)[2 * b], n = ((const int*)p.scratch)[2 * b + 1];
    const int NKV = p.NH / p.gqa, kvh = h / p.gqa, r = tk * p.gqa + h - kvh * p.gqa, X = NKV * ngrp;
    ns = n < 0 ? -n : n;
    if (ns < 2) return;
    const long long slot = (long long)X * 16 * (HDr + 2);
    base = p.scratch + dec_meta_floats(p) + ((long long)slot0 * X + (r >> 4) * NKV + kvh) * 16 * (HDr + 2) + (r & 15) * (HDr + 2);
    rest = n < 0 ? -slot : 0;
    step = 2 * slot;
  }
  // the splits in chunks of NC (2, 4 or 8, at least the split count up to 8) whose loads are all
  // issued before any is used (indices past the last split repeat it and are not used): one
  // memory latency per chunk (a batch-1 decode of 21 splits took 12 us here with one load per step);
  // the sums run in split order, scaled where a chunk raises the maximum
  auto rec = [&](int s) {
    s = min(s, ns - 1);
    return base + s * step + (STREAM && s > 0 ? rest : 0);
  };
  float gm = -INFINITY, l = 0.0f, acc = 0.0f;
  auto merge = [&](auto chunk) {
    constexpr int kC = decltype(chunk)::value;
    for (int s0 = 0; s0 < ns; s0 += kC) {
      float m[kC], ls[kC], a[kC];
#pragma unroll
      for (int u = 0; u < kC; u++) {
        const float* ps = rec(s0 + u);
        m[u] = ps[0];
        ls[u] = ps[1];
        a[u] = ps[2 + dc];
      }
      float nm = gm;
#pragma unroll
      for (int u = 0; u < kC; u++)
        if (s0 + u < ns) nm = fmaxf(nm, m[u]);
      if (nm == -INFINITY) continue;   // no key so far
      const float keep = exp2_fast(gm - nm);
      l *= keep;
      acc *= keep;
      gm = nm;
#pragma unroll
      for (int u = 0; u < kC; u++) {
        if (s0 + u < ns) {
          const float w = exp2_fast(m[u] - gm);
          l += w * ls[u];
          acc += w * a[u];
        }
      }
    }
  };
  if (STREAM && ns == 2)
    merge(std::integral_constant<int, 2>{});
  else
    merge(std::integral_constant<int, NC>{});
  const bool ok = gm != -INFINITY && l > 0.0f;
  if (d < HDr) ((T*)p.o)[((long long)row * p.NH + h) * HDr + d] = (T)(ok ? acc / l : 0.0f);
  if (p.lse_out && d == 0) p.lse_out[(long long)row * p.NH + h] = ok ? gm * kLn2 + __logf(l) : -INFINITY;
}

// write new_k (rotary applied) / new_v at positions ctx_len[b]+tk: grid (batch*nq, NKV), block HD
template <typename T, int HD>
__global__ __launch_bounds__(256) void dec_append_kernel(FableDecParams p, const T* nk, const T* nv, int page_shift) {
  __shared__ float ks[HD];
  // one thread per column of the kernel width HD; rows are p.HD <= HD long
  const int b = blockIdx.x / p.nq, tk = blockIdx.x % p.nq, kvh = blockIdx.y, d = threadIdx.x;
  const int NKV = p.NH / p.gqa, HDr = p.HD;
  const int pos = p.ctx_len[b] + tk;
  const bool ok = pos >= 0 && (pos >> page_shift) < p.max_blocks && d < HDr;
  const long long src = ((long long)(b * p.nq + tk) * NKV + kvh) * HDr;
  ks[d] = d < HDr ? (float)nk[src + d] : 0.0f;
  __syncthreads();
  if (p.rotary) {
    const int rdim = p.rotary_dim > 0 ? p.rotary_dim : HDr, half = rdim / 2;
    const int rp = (p.rotary_pos ? p.rotary_pos[b] : p.ctx_len[b]) + tk;
    const bool act = d < half;
    const int ia = p.rotary == 1 ? d : 2 * d, ib = p.rotary == 1 ? d + half : 2 * d + 1;
    float x = 0.0f, y = 0.0f, c = 0.0f, s = 0.0f;
    if (act) {
      c = p.cos[(long long)rp * half + d];
      s = p.sin[(long long)rp * half + d];
      x = ks[ia];
      y = ks[ib];
    }
    __syncthreads();
    if (act) {
      ks[ia] = x * c - y * s;
      ks[ib] = y * c + x * s;
    }
    __syncthreads();
  }
  if (!ok) return;
  const int j = pos >> page_shift, blk = p.block_table ? p.block_table[(long long)b * p.max_blocks + j] : b * p.max_blocks + j;
  const long long dst = (((long long)blk * p.page + (pos & (p.page - 1))) * NKV + kvh) * HDr + d;
  ((T*)p.Kc)[dst] = (T)ks[d];
  ((T*)p.Vc)[dst] = nv[src + d];
}

// row groups of 16 per (sequence, K/V head)
static int dec_groups(const FableDecParams& p) { return (int)(((long long)p.nq * p.gqa + 15) / 16); }

// Parts of a call (DecShare): one workgroup per CU (more in flight per CU read a batch of alike
// sequences slower: C4 0.96x with two, 0.86x with three), or two where the (K/V head, row group) count
// leaves more than an eighth of the CUs out of a round of one.
static int dec_parts(const FableDecParams& p) {
  const long long X = (long long)(p.NH / p.gqa) * dec_groups(p);
  long long parts = 256 / X;
  if (parts * X < 224) parts = (512 + X - 1) / X;
  const long long units = (long long)p.batch * (((long long)p.max_blocks * p.page + kUnit - 1) / kUnit + 1);
  parts = parts < units ? parts : units;
  return parts > 1 ? (int)parts : 1;
}
// workgroups per (K/V head, row group) (DecShare::init)
static int dec_share_wgs(const FableDecParams& p) { return p.batch <= dec_parts(p) ? dec_parts(p) : 2 * dec_parts(p); }
// scratch: two records of 16 rows per workgroup
static long long dec_share_bytes(const FableDecParams& p) {
  return (dec_meta_floats(p) + (long long)dec_share_wgs(p) * 2 * (p.NH / p.gqa) * dec_groups(p) * 16 * (p.HD + 2)) * 4;
}

template <typename T, int HD>
static int launch_dec_partial(const FableDecParams& p, dim3 grid, int page_shift, int flags, int parts, hipStream_t st, const void* nk,
                              const void* nv) {
  const bool feat = p.softcap > 0.0f || p.alibi != nullptr, spt = p.page >= 16;
  auto go = [&](auto ft, auto sp, auto sh) {
    DecArgs a;
    (FableDecParams&)a = p;
    a.nk = nk;
    a.nv = nv;
    a.table = p.block_table ? p.block_table : p.ctx_len;
    a.tmask = p.block_table ? -1 : 0;
    a.page_shift = page_shift;
    a.ngrp = dec_groups(p);
    a.flags = flags;
    a.parts = parts;
    a.nkv = p.NH / p.gqa;
    hipLaunchKernelGGL((dec_partial_kernel<T, HD, decltype(ft)::value, decltype(sp)::value, decltype(sh)::value>), grid, dim3(256), 0, st, a);
  };
  using Y = std::integral_constant<bool, true>;
  using N = std::integral_constant<bool, false>;
  if (parts > 0)   // (pages of at least 16 rows: dec_shares)
    feat ? go(Y{}, Y{}, Y{}) : go(N{}, Y{}, Y{});
  else if (feat)
    spt ? go(Y{}, Y{}, N{}) : go(Y{}, N{}, N{});
  else
    spt ? go(N{}, Y{}, N{}) : go(N{}, N{}, N{});
  return launch_status("fable_attn_dec (partial)");
}

template <typename T, int HD>
static int launch_dec_append(const FableDecParams& p, hipStream_t st, const void* nk, const void* nv) {
  hipLaunchKernelGGL((dec_append_kernel<T, HD>), dim3(p.batch * p.nq, p.NH / p.gqa), dim3(HD), 0, st, p, (const T*)nk, (const T*)nv,
                     __builtin_ctz((unsigned)p.page));
  return launch_status("fable_attn_dec (append)");
}
// Whether the partial kernel writes the new key itself: one token per sequence, whose row no other
// sequence can read. With a block table two sequences may name one page (drafted tokens laid out as
// batch rows of successive lengths, a cache row given twice), and then a workgroup that reads the row
// must find it written: by a kernel ahead, as for several tokens. (v is copied in 16-byte pieces.)
template <typename T>
static bool dec_fuses_append(const FableDecParams& p, const void* nv) {
  return !std::is_same<T, float>::value && p.nq == 1 && (!p.block_table || p.batch == 1) && ((uintptr_t)nv & 15) == 0;
}

template <typename T, int HD>
static int launch_dec(const FableDecParams& p, hipStream_t st, const void* nk, const void* nv) {
  const int page_shift = __builtin_ctz((unsigned)p.page);
  const int NKV = p.NH / p.gqa;
  const int ngrp = (p.gqa + 15) / 16;
  const bool fuse = dec_fuses_append<T>(p, nv);
  if (nk && !fuse)
    if (int rc = launch_dec_append<T, HD>(p, st, nk, nv)) return rc;
  const bool feat = p.softcap > 0.0f || p.alibi != nullptr;
  if constexpr (std::is_same<T, float>::value) {
    const dim3 grid(NKV * ngrp, p.batch * p.nq, p.nsplit);
    if (feat)
      hipLaunchKernelGGL((dec_partial_f32_kernel<HD, true>), grid, dim3(256), 0, st, p, page_shift, ngrp, nk ? 1 : 0);
    else
      hipLaunchKernelGGL((dec_partial_f32_kernel<HD, false>), grid, dim3(256), 0, st, p, page_shift, ngrp, nk ? 1 : 0);
  } else {
    // one split: the partial kernel writes the output and LSE, and no combine is launched
    const int flags = (nk ? kDecAppend : 0) | (p.nsplit == 1 ? kDecFinal : 0);
    if (int rc = launch_dec_partial<T, HD>(p, dim3(NKV * dec_groups(p), p.batch, p.nsplit), page_shift, flags, 0, st, fuse ? nk : nullptr, nv)) return rc;
    if (p.nsplit == 1) return FA_OK;
  }
  if (int rc = launch_status("fable_attn_dec (partial)")) return rc;
  const dim3 cg(p.batch * p.nq, p.NH);
  if (p.nsplit <= 2)
    hipLaunchKernelGGL((dec_combine_kernel<T, HD, 2>), cg, dim3(HD), 0, st, p, 0);
  else if (p.nsplit <= 4)
    hipLaunchKernelGGL((dec_combine_kernel<T, HD, 4>), cg, dim3(HD), 0, st, p, 0);
  else
    hipLaunchKernelGGL((dec_combine_kernel<T, HD, 8>), cg, dim3(HD), 0, st, p, 0);
  return launch_status("fable_attn_dec (combine)");
}

// the call with its shares worked out on the device (p.nsplit 0)
template <typename T, int HD>
static int launch_dec_share(const FableDecParams& p, hipStream_t st, const void* nk, const void* nv) {
  const int ngrp = dec_groups(p), X = p.NH / p.gqa * ngrp, parts = dec_parts(p);
  const bool fuse = dec_fuses_append<T>(p, nv);
  if (nk && !fuse)
    if (int rc = launch_dec_append<T, HD>(p, st, nk, nv)) return rc;
  if (int rc = launch_dec_partial<T, HD>(p, dim3((unsigned)X, (unsigned)dec_share_wgs(p)), __builtin_ctz((unsigned)p.page), nk ? kDecAppend : 0, parts,
                                         st, fuse ? nk : nullptr, nv))
    return rc;
  hipLaunchKernelGGL((dec_combine_kernel<T, HD, 8, true>), dim3(p.batch * p.nq, p.NH), dim3(HD), 0, st, p, ngrp);
  return launch_status("fable_attn_dec (combine)");
}

// fp16/bf16: every head dim that is a multiple of 8 up to 256 runs in the kernel of the next
// multiple of 32 (64 at least: the K slice swizzle needs 8 chunks per row) with zero columns
// past it. The loads skip those columns' bytes, so HBM traffic is that of the real head dim.
// fp32 runs in kernels of width 64, 128 and 256, the same way.
template <typename T, int HD>
static int launch_dec_any(const FableDecParams& p, hipStream_t st, const void* nk, const void* nv) {
  if constexpr (!std::is_same<T, float>::value)
    if (p.nsplit == 0) return launch_dec_share<T, HD>(p, st, nk, nv);
  return launch_dec<T, HD>(p, st, nk, nv);
}
template <typename T>
static int dec_dispatch(const FableDecParams& p, hipStream_t st, const void* nk, const void* nv) {
  constexpr bool f32 = std::is_same<T, float>::value;
  if (p.HD <= 0 || p.HD > 256 || p.HD % 8)
    return fail(FA_ERR_HEADDIM, "fable_attn_dec: head_dim=%d has no kernel (multiples of 8 up to 256)", p.HD);
  if constexpr (f32) {
    if (p.HD <= 64) return launch_dec_any<T, 64>(p, st, nk, nv);
    if (p.HD <= 128) return launch_dec_any<T, 128>(p, st, nk, nv);
    return launch_dec_any<T, 256>(p, st, nk, nv);
  } else {
    switch (p.HD <= 64 ? 2 : (p.HD + 31) / 32) {
      case 2: return launch_dec_any<T, 64>(p, st, nk, nv);
      case 3: return launch_dec_any<T, 96>(p, st, nk, nv);
      case 4: return launch_dec_any<T, 128>(p, st, nk, nv);
      case 5: return launch_dec_any<T, 160>(p, st, nk, nv);
      case 6: return launch_dec_any<T, 192>(p, st, nk, nv);
      case 7: return launch_dec_any<T, 224>(p, st, nk, nv);
      default: return launch_dec_any<T, 256>(p, st, nk, nv);
    }
  }
}

}  // namespace fa

// Split count from a model of the partial kernel as a stream of workgroup rounds: one
// workgroup per CU is resident (256 CUs), the cache read saturates HBM once ~168 workgroups
// stream together, and each split pays a fixed cost of about 64 keys (prologue, partial
// write, combine). Time of a round of t workgroups ~ t * (keys per split + 64) / min(t, 168);
// the smallest n within the minimum wins. At least 256 keys per split, n in [1, 512].
// On the C4 shape (128 groups, 32768 keys) the model ranks n = 1, 2, 3, 4 as measured on
// MI355X (474, 371, 414, 375 us). Reference heuristic (72 CUs): package/csrc/dispatch.cpp:182-200.
extern "C" int fa_decode_num_splits(int batch, int nq, int NH, int gqa, int64_t ctx_bound, int hint) {
  if (hint > 0) return hint > 512 ? 512 : hint;
  constexpr long long kSlots = 256, kSat = 168, kSplitCost = 64;
  const int g = gqa > 0 ? gqa : 1;
  long long groups = (long long)batch * (nq > 0 ? nq : 1) * (NH / g > 0 ? NH / g : 1) * ((g + 15) / 16);
  if (groups < 1) groups = 1;
  const long long ctx = ctx_bound > 1 ? ctx_bound : 1;
  long long maxn = (ctx + 255) / 256;
  maxn = maxn < 1 ? 1 : (maxn > 512 ? 512 : maxn);
  int best = 1;
  double best_cost = 0.0;
  for (long long n = 1; n <= maxn; n++) {
    const double per = (double)((ctx + n - 1) / n + kSplitCost);
    const long long wgs = groups * n, full = wgs / kSlots, tail = wgs % kSlots;
    double cost = (double)full * kSlots * per / kSat;
    if (tail) cost += (double)tail * per / (double)(tail < kSat ? tail : kSat);
    if (n == 1 || cost < best_cost * 0.995) {
      best = (int)n;
      best_cost = cost;
    }
  }
  // A choice that leaves CUs idle in its one round: with few groups each workgroup streams a
  // long span alone, below the rate the model's saturation point assumes, so fill the round
  // while every split keeps at least kFillKeys keys (batch 1, 8 kv heads, 32768 keys: 21 -> 32
  // splits, partial kernel 30.0 -> 24.5 us)
  constexpr long long kFillKeys = 512;
  const long long fill = kSlots / groups;
  if ((long long)best * groups < kSlots && fill > best && fill <= maxn && (ctx + fill - 1) / fill >= kFillKeys)
    best = (int)fill;
  return best;
}

// Whether a call reads or writes p.scratch: with one split the fp16/bf16 partial kernel writes the
// output and LSE itself and no combine runs; fp32 always combines through the scratch.
static bool dec_uses_scratch(const FableDecParams& p, int dtype) { return p.nsplit != 1 || dtype == FA_F32; }

extern "C" int fable_attn_dec(FableDecParams p, int dtype, void* stream, const void* new_k, const void* new_v) {
  using namespace fa;
  if (!p.q || !p.Kc || !p.Vc || !p.block_table || !p.o || !p.ctx_len)
    return fail(FA_ERR_ARG, "fable_attn_dec: null pointer");
  if (!p.scratch && dec_uses_scratch(p, dtype))
    return fail(FA_ERR_ARG, "fable_attn_dec: null scratch (needed unless nsplit == 1 with fp16/bf16)");
  return dec_checked(p, dtype, stream, new_k, new_v);
}

// ------------------------------------------------------------------ decode without allocation
// The split partials live in a device array of fixed size that the library owns (one copy per
// GPU, held until the process ends), for callers that cannot allocate: code under HIP graph
// capture, tight serving loops, harnesses that forbid hipMalloc. In host code `dec_scratch`
// names a host-side stand-in, not device memory: its device address on the current GPU comes
// from hipGetSymbolAddress, once per device, and only that address is ever passed to a kernel.
// Every partial slot is written before the combine reads it, so nothing needs clearing between
// calls; calls that overlap on one GPU (two streams, or a graph replay beside an eager call)
// race on the array and must be serialised by the caller.
namespace {

constexpr long long kDecScratchFloats = 4ll << 20;  // 16 MiB
static __device__ __align__(256) float dec_scratch[kDecScratchFloats];

constexpr int kMaxDevices = 64;
std::mutex g_dec_scratch_mu;
float* g_dec_scratch_ptr[kMaxDevices] = {};

// device address of dec_scratch on the GPU of `stream` (which must be the current device)
int dec_scratch_ptr(void* stream, float** out) {
  using fa::fail;
  int cur = -1;
  if (hipGetDevice(&cur) != hipSuccess || cur < 0 || cur >= kMaxDevices)
    return fail(FA_ERR_LAUNCH, "fable_attn_dec_noalloc: no current device (%d)", cur);
  if (stream) {
    hipDevice_t sdev = -1;
    if (hipStreamGetDevice((hipStream_t)stream, &sdev) != hipSuccess)
      return fail(FA_ERR_ARG, "fable_attn_dec_noalloc: the stream's device is unknown");
    if (sdev != cur)
      return fail(FA_ERR_ARG, "fable_attn_dec_noalloc: the stream belongs to device %d, the current "
                              "device is %d (make the stream's device current)", (int)sdev, cur);
  }
  std::lock_guard<std::mutex> lock(g_dec_scratch_mu);
  if (!g_dec_scratch_ptr[cur]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(dec_scratch));
    if (e != hipSuccess || !ptr)
      return fail(FA_ERR_LAUNCH, "fable_attn_dec_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
    g_dec_scratch_ptr[cur] = (float*)ptr;
  }
  *out = g_dec_scratch_ptr[cur];
  return FA_OK;
}

}  // namespace

extern "C" int64_t fable_attn_dec_noalloc_max_floats(void) { return kDecScratchFloats; }

extern "C" int fable_attn_dec_noalloc(FableDecParams p, int dtype, void* stream, const void* new_k,
                                      const void* new_v) {
  using namespace fa;
  if (!p.q || !p.Kc || !p.Vc || !p.block_table || !p.o || !p.ctx_len)
    return fail(FA_ERR_ARG, "fable_attn_dec_noalloc: null pointer");
  if (p.batch <= 0) return FA_OK;
  if (p.NH <= 0) return fail(FA_ERR_ARG, "fable_attn_dec_noalloc: NH=%d", p.NH);
  if (p.nsplit < 1 || p.nsplit > 512) return fail(FA_ERR_ARG, "fable_attn_dec_noalloc: nsplit=%d", p.nsplit);
  if (p.HD <= 0) return fail(FA_ERR_HEADDIM, "fable_attn_dec_noalloc: head_dim=%d", p.HD);
  // one fp16/bf16 split never touches the array: no size limit then
  const long long need = (long long)p.batch * (p.nq < 1 ? 1 : p.nq) * p.NH * p.nsplit * (p.HD + 2);
  if (dec_uses_scratch(p, dtype) && need > kDecScratchFloats)
    return fail(FA_ERR_ARG, "fable_attn_dec_noalloc: batch*nq*NH*nsplit*(HD+2) = %lld floats of split "
                            "partials exceed the fixed %lld (lower nsplit, or use fable_attn_dec with a "
                            "caller-allocated scratch)", need, kDecScratchFloats);
  if (int rc = dec_scratch_ptr(stream, &p.scratch)) return rc;
  return dec_checked(p, dtype, stream, new_k, new_v);
}

namespace fa {

// ------------------------------------------------------------------ many new tokens at once
// A call whose new tokens give a K/V head at least kTileRows rows (tokens x heads of its group)
// runs on the tile kernel of the forward (fwd_kernel over FwdPaged): the decode kernel reads a
// sequence's K/V once per new token, which for a chunk of a prompt is all its time. Appending 512
// rotated tokens to each of two requests with 1000-7000 cached keys (Hq 32 / Hk 8, D 128, bf16):
// 1710 us -> 197 us. At 64 rows the tile kernel takes 0.11-0.92x the decode kernel's time (batch 1
// to 32, 500 to 32000 keys, D 64 to 256; 16 tokens of 4 heads over 32000 keys 227 -> 51 us), at
// 512 rows 0.07-0.39x. (Where a table for many keys holds a few hundred, batches of 1 to 4 with up to 256
// rows pay the three kernels' latency: 64 rows over 600 keys under a table of 32768, batch 1, 20 us, 14 before.
// The keys are not known here.)
// With few K/V heads and sequences the tile kernel has few tiles, each in at most 32 splits, and the decode
// kernel up to 512 splits of every 16 rows: up to kTileStreams (sequence, K/V head, 16 rows) the decode kernel
// keeps the call. One token, 64 heads of one K/V head, D 128: batch 1, 8000 keys 18 us and 24 on the tiles,
// 32000 28 and 49, batch 4 26 and 25, 49 and 52; past it batch 16, 8000 keys 46 and 35. 128 heads: batch 2,
// 32000 keys 49 and 56, batch 4 82 and 57.
constexpr int kTileRows = 64, kTileStreams = 16;
// (A window of 0 keys, which leaves no key visible, has no form in the forward's bounds: the decode
// kernel serves it; so does it tables of 2^31 entries, and pages of 2^31 elements, and more.)
static bool dec_uses_tiles(const FableDecParams& p, int dtype) {
  if (p.gqa <= 0 || (long long)p.batch * (p.NH / p.gqa) * dec_groups(p) <= kTileStreams) return false;
  return (dtype == FA_F16 || dtype == FA_BF16) && p.gqa > 0 && (long long)p.nq * p.gqa >= kTileRows && p.page >= 16 &&
         (long long)p.batch * p.max_blocks <= 0x7FFFFFFF && p.max_blocks < (1 << 29) && (long long)(p.NH / p.gqa) * p.HD * p.page <= 0x7FFFFFFF && p.window != 0 && p.HD > 0 && p.HD <= 256 && p.HD % 8 == 0;
}

// Before the tile kernel, gridDim.y workgroups per new token: the token's k (rotated) and v rows go to
// the cache, and its q rows, rotated in fp32, to two 16-bit tensors whose sum is the rotated q to
// 2^-16 (bf16) or 2^-22 (fp16) of its value, as the decode kernel carries it; in fp16 no better than
// 2^-25 absolute (the low part of values under 2^-3 is subnormal). (One workgroup per
// token walked 64 tokens of 64 + 8 heads in 14.5 us; now 4.6.)
template <typename T>
__global__ __launch_bounds__(256) void dec_prep_kernel(FableDecParams p, const T* nk, const T* nv, T* qhi, T* qlo, int page_shift) {
  const int b = blockIdx.x / p.nq, tk = blockIdx.x % p.nq, NKV = p.NH / p.gqa, HDr = p.HD;
  const int rdim = p.rotary ? (p.rotary_dim > 0 ? p.rotary_dim : HDr) : 0, half = rdim / 2;
  const int ctx = p.ctx_len[b], pos = ctx + tk;
  const long long rp = (p.rotary_pos ? p.rotary_pos[b] : ctx) + tk;
  const bool ok = nk && pos >= 0 && (pos >> page_shift) < p.max_blocks;
  long long dst = 0;
  if (ok) {
    const int j = pos >> page_shift, blk = p.block_table ? p.block_table[(long long)b * p.max_blocks + j] : b * p.max_blocks + j;
    dst = ((long long)blk * p.page + (pos & (p.page - 1))) * NKV * HDr;
  }
  const long long tok = (long long)b * p.nq + tk;
  const T* q = (const T*)p.q + tok * p.NH * HDr;
  const int t0 = blockIdx.y * 256 + threadIdx.x, step = gridDim.y * 256;
  const int nh = qhi ? p.NH : 0, total = nh + (ok ? NKV : 0);  // heads to rotate: q, then k
  // rotated pairs: item i is pair i % half of head i / half
  for (int i = t0; i < total * half; i += step) {
    const int g = i / half, j = i - g * half;
    const float c = p.cos[rp * half + j], s = p.sin[rp * half + j];
    const int ia = p.rotary == 1 ? j : 2 * j, ib = p.rotary == 1 ? j + half : 2 * j + 1;
    const T* src = g < nh ? q + (long long)g * HDr : nk + (tok * NKV + g - nh) * HDr;
    const float x = (float)src[ia], y = (float)src[ib];
    const float xr = x * c - y * s, yr = y * c + x * s;
    if (g < nh) {
      const long long o = (tok * p.NH + g) * HDr;
      const T xh = (T)xr, yh = (T)yr;
      qhi[o + ia] = xh;
      qhi[o + ib] = yh;
      qlo[o + ia] = (T)(xr - (float)xh);
      qlo[o + ib] = (T)(yr - (float)yh);
    } else {
      T* kd = (T*)p.Kc + dst + (long long)(g - nh) * HDr;
      kd[ia] = (T)xr;
      kd[ib] = (T)yr;
    }
  }
  // columns past the rotary width, and v
  const int rest = HDr - rdim;
  for (int i = t0; i < total * rest; i += step) {
    const int g = i / rest, d = rdim + i - g * rest;
    if (g < nh) {
      const long long o = (tok * p.NH + g) * HDr + d;
      qhi[o] = q[(long long)g * HDr + d];
      qlo[o] = (T)0.0f;
    } else {
      ((T*)p.Kc)[dst + (long long)(g - nh) * HDr + d] = nk[(tok * NKV + g - nh) * HDr + d];
    }
  }
  if (ok)
    for (int i = t0; i < NKV * HDr / 8; i += step)
      *(u32x4*)((T*)p.Vc + dst + 8 * i) = *(const u32x4*)(nv + tok * NKV * HDr + 8 * i);
}

// the forward's parameters of a call on the tile kernel
static void dec_tile_params(const FableDecParams& p, bool append, FableFwdParams& f, FwdPaged& pg) {
  const int64_t NKV = p.NH / p.gqa, D = p.HD;
  f = FableFwdParams{};
  f.Q = p.q;
  f.K = p.Kc;
  f.V = p.Vc;
  f.O = p.o;
  f.LSE = p.lse_out;
  f.sQ = f.sO = fa_strides{p.nq * p.NH * D, D, p.NH * D};
  f.sK = f.sV = fa_strides{0, D, NKV * D};
  f.SQ = p.nq;
  const long long room = (long long)p.max_blocks * p.page;
  f.SK = room < 0x7FFFFFFF ? (int)room : 0x7FFFFFFF;  // the most a sequence can hold
  f.HD = p.HD;
  f.NH = p.NH;
  f.gqa = p.gqa;
  f.scale = p.scale;
  f.softcap = p.softcap;
  f.win_left = p.window >= 0 ? p.window - 1 : -1;
  f.win_right = -1;
  f.alibi_slopes = p.alibi;
  f.causal = append;
  f.batch = p.batch;
  f.lse_sb = (int64_t)p.nq * p.NH;
  f.lse_sh = 1;
  pg = FwdPaged{p.block_table ? p.block_table : p.ctx_len, p.block_table ? -1 : 0, p.max_blocks, __builtin_ctz((unsigned)p.page), p.page * NKV * D, p.page * NKV * D, p.ctx_len,
                append ? 1 : 0, p.leftpad, nullptr, p.NH};
}

static long long align256(long long x) { return (x + 255) / 256 * 256; }

// bytes of one part of a rotated q in the workspace
static long long dec_q_bytes(const FableDecParams& p) {
  return p.rotary ? align256((long long)p.batch * p.nq * p.NH * p.HD * 2) : 0;
}

template <typename T>
static int launch_dec_tiles(const FableDecParams& p, int dtype, int nsplit, char* ws, long long ws_bytes, hipStream_t st, const void* nk,
                            const void* nv) {
  FableFwdParams f;
  FwdPaged pg;
  dec_tile_params(p, nk != nullptr, f, pg);
  const long long qb = dec_q_bytes(p);
  if (2 * qb > ws_bytes) return fail(FA_ERR_ARG, "fable_attn_dec_ws: workspace of %lld bytes, %lld needed", ws_bytes, 2 * qb);
  if (p.rotary || nk) {
    T* qhi = p.rotary ? (T*)ws : nullptr;
    T* qlo = p.rotary ? (T*)(ws + qb) : nullptr;
    // (few tokens: workgroups for every 256 items of a token's walk; many fill the chip with one each)
    const long long tokens = (long long)p.batch * p.nq, items = (long long)(p.NH + p.NH / p.gqa) * p.HD / 2;
    long long slices = 2048 / tokens < (items + 255) / 256 ? 2048 / tokens : (items + 255) / 256;
    slices = slices > 1 ? slices : 1;
    hipLaunchKernelGGL((dec_prep_kernel<T>), dim3((unsigned)tokens, (unsigned)slices), dim3(256), 0, st, p, (const T*)nk, (const T*)nv,
                       qhi, qlo, pg.page_shift);
    if (int rc = launch_status("fable_attn_dec (append)")) return rc;
    if (p.rotary) {
      f.Q = qhi;
      pg.qlo = qlo;
    }
  }
  FwdWs fw{ws ? ws + 2 * qb : nullptr, ws_bytes - 2 * qb, false, 0, nsplit};
  return launch_fwd_paged(f, pg, dtype, p.rotary != 0, st, fw);
}

// the argument checks of the decode entry points (nq below 1 becomes 1)
static int dec_check(FableDecParams& p, const void* new_k, const void* new_v) {
  if (p.page <= 0 || (p.page & (p.page - 1))) return fail(FA_ERR_ARG, "fable_attn_dec: page=%d is not a power of two", p.page);
  if (p.NH <= 0 || p.gqa <= 0 || p.NH % p.gqa) return fail(FA_ERR_ARG, "fable_attn_dec: NH=%d gqa=%d", p.NH, p.gqa);
  if (p.nsplit < 1 || p.nsplit > 512) return fail(FA_ERR_ARG, "fable_attn_dec: nsplit=%d", p.nsplit);
  if (p.nq < 1) p.nq = 1;
  if ((new_k == nullptr) != (new_v == nullptr)) return fail(FA_ERR_ARG, "fable_attn_dec: new_k and new_v go together");
  if (p.rotary && (!p.cos || !p.sin)) return fail(FA_ERR_ARG, "fable_attn_dec: rotary needs cos and sin");
  if (p.rotary && (p.rotary_dim < 0 || p.rotary_dim > p.HD || p.rotary_dim % 2)) return fail(FA_ERR_ARG, "fable_attn_dec: rotary_dim=%d", p.rotary_dim);
  return FA_OK;
}

// the checks and dispatch shared by fable_attn_dec and fable_attn_dec_noalloc
static int dec_checked(FableDecParams p, int dtype, void* stream, const void* new_k, const void* new_v) {
  if (int rc = dec_check(p, new_k, new_v)) return rc;
  if (p.batch <= 0) return FA_OK;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case FA_F16: return dec_dispatch<_Float16>(p, st, new_k, new_v);
    case FA_BF16: return dec_dispatch<__bf16>(p, st, new_k, new_v);
    case FA_F32: return dec_dispatch<float>(p, st, new_k, new_v);
    default: return fail(FA_ERR_DTYPE, "fable_attn_dec: dtype %d not implemented (fp16/bf16/fp32)", dtype);
  }
}

}  // namespace fa

// fable_attn_dec with one workspace for whatever the call needs. p.nsplit: the caller's count (0:
// the library's choice).
// Whether the shares are worked out on the device: fp16/bf16, no count of the caller's, pages of at
// least 16 rows, a table that can hold kShareBytes of keys and values, and a batch that equal
// splits would not spread evenly over the parts (more sequences than parts, or a count that
// does not divide them). The shares take 1-2 us (ahead of the first load, and in a combine that is always
// launched), which short sequences under a table for long ones do not win back (3 x 500 keys, Hq 32 / Hk 8,
// D 128: 10.2 us in equal splits, 11.6 shared; 24 x 500 15.8 and 19.0; 64 x 500 26.5 and 29.1), while long ones
// of unequal lengths gain more (12 of 750-8000 keys 65.6 and 39.7, 24 of 333-8000 123 and 78, 48 x 64-8192
// of Hq 64 / Hk 8 155 and 135): the lengths are not known here, the size of the table is. A batch that divides the
// parts keeps equal splits, which share sequences of one length evenly without (16 x 32768 keys 311 and 314 us)
// but leave unequal ones waiting for the longest (eight of 1000 to 16000 keys 68 us, 53 if shared).
constexpr long long kShareBytes = 128LL << 20;
static bool dec_shares(const FableDecParams& p, int dtype) {
  if (dtype == FA_F32 || p.nsplit > 0 || p.batch < 2 || p.gqa <= 0 || p.page < 16) return false;
  if ((long long)p.batch * p.max_blocks * p.page * (p.NH / p.gqa) * p.HD * 4 < kShareBytes) return false;
  const int parts = fa::dec_parts(p);
  return p.batch > parts || parts % p.batch != 0;
}
// splits per sequence otherwise: its rows are packed into dec_groups groups
static int dec_fixed_splits(const FableDecParams& p, int dtype) {
  const int64_t bound = (int64_t)p.max_blocks * p.page;
  return dtype == FA_F32 ? fa_decode_num_splits(p.batch, p.nq, p.NH, p.gqa, bound, p.nsplit)
                         : fa_decode_num_splits(p.batch, fa::dec_groups(p), p.NH / p.gqa, 1, bound, p.nsplit);
}

extern "C" int64_t fable_attn_dec_ws_bytes(FableDecParams p, int dtype, int append) {
  using namespace fa;
  if (p.nq < 1) p.nq = 1;
  if (p.NH <= 0 || p.gqa <= 0 || p.NH % p.gqa || p.batch <= 0 || p.HD <= 0 || p.page <= 0 || p.max_blocks < 0) return 0;
  if (dec_uses_tiles(p, dtype)) {
    FableFwdParams f;
    FwdPaged pg;
    dec_tile_params(p, append != 0, f, pg);
    FwdWs fw{nullptr, 0, true, 0, p.nsplit};
    if (launch_fwd_paged(f, pg, dtype, p.rotary != 0, nullptr, fw) != FA_OK) return -1;
    return 2 * dec_q_bytes(p) + fw.need;
  }
  if (dec_shares(p, dtype)) return dec_share_bytes(p);
  p.nsplit = dec_fixed_splits(p, dtype);
  return dec_uses_scratch(p, dtype) ? (int64_t)p.batch * p.nq * p.NH * p.nsplit * (p.HD + 2) * 4 : 0;
}

extern "C" int fable_attn_dec_ws(FableDecParams p, int dtype, void* ws, int64_t ws_bytes, void* stream_, const void* new_k,
                                 const void* new_v) {
  using namespace fa;
  if (!p.q || !p.Kc || !p.Vc || !p.o || !p.ctx_len) return fail(FA_ERR_ARG, "fable_attn_dec_ws: null pointer");
  if (p.nq < 1) p.nq = 1;
  const bool tiles = dec_uses_tiles(p, dtype), share = !tiles && dec_shares(p, dtype);
  if (!p.block_table && dtype == FA_F32) return fail(FA_ERR_ARG, "fable_attn_dec_ws: null block_table (fp32)");
  const int hint = p.nsplit;
  p.nsplit = 1;
  if (int rc = dec_check(p, new_k, new_v)) return rc;
  if (p.batch <= 0) return FA_OK;
  if (tiles)
    return dtype == FA_F16 ? launch_dec_tiles<_Float16>(p, dtype, hint, (char*)ws, ws_bytes, (hipStream_t)stream_, new_k, new_v)
                           : launch_dec_tiles<__bf16>(p, dtype, hint, (char*)ws, ws_bytes, (hipStream_t)stream_, new_k, new_v);
  long long need;
  if (share) {
    need = dec_share_bytes(p);
  } else {
    p.nsplit = hint;
    p.nsplit = dec_fixed_splits(p, dtype);
    need = dec_uses_scratch(p, dtype) ? (long long)p.batch * p.nq * p.NH * p.nsplit * (p.HD + 2) * 4 : 0;
  }
  if (need > 0 && (!ws || ws_bytes < need))
    return fail(FA_ERR_ARG, "fable_attn_dec_ws: workspace of %lld bytes, %lld needed", (long long)ws_bytes, need);
  p.scratch = (float*)ws;
  if (!share) return dec_checked(p, dtype, stream_, new_k, new_v);
  p.nsplit = 0;
  switch (dtype) {
    case FA_F16: return dec_dispatch<_Float16>(p, (hipStream_t)stream_, new_k, new_v);
    case FA_BF16: return dec_dispatch<__bf16>(p, (hipStream_t)stream_, new_k, new_v);
    default: return fail(FA_ERR_DTYPE, "fable_attn_dec_ws: dtype %d not implemented (fp16/bf16/fp32)", dtype);
  }
}
