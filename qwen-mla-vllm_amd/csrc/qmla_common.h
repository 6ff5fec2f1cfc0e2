// Shared by the decode translation units of libqmla.so: the kernel parameter block, the output
// descriptor of one token range, and the split of a launch into token ranges (fixed splits or the
// balanced plan).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "qmla.h"
#include "qmla_device.h"

namespace qmla {

constexpr int PLAN_TILE = 64;  // balancing granularity of the balanced plan (tokens)
// plan tiles the balanced plan charges per request switch (see plan_tiles), per kernel family: the
// warp-specialized and row-owner decode, for a piece's query load and output write, the per-group and
// column-split kernels (none). At 1 / 2 / 3 tiles, whole call, alternating runs: GLA-g2 B 48 x 4 168.2 /
// 167.2 / 168.7 us, verify B 64 x 4 358.8 / 356.8 / 356.5, bf16 B 64 221.2 / 220.6 / 222.6, the FP8 B 128
// headline the same; 4 layers of 23 rank-768 requests 185.8 / 175.2 / 165.0
constexpr int kPlanSwitchWs = 2, kPlanSwitchRo = 2, kPlanSwitchOther = 0;

struct KParams {
  const __bf16* q_nope;
  int64_t qn_sr, qn_sh;
  const __bf16* q_pe;
  int64_t qp_sr, qp_sh;
  const char* kv;
  int64_t page_stride_b, token_stride_b;  // bytes
  int page_size;
  uint32_t page_mul;    // x / page_size = (x * page_mul) >> page_sh for 0 <= x < 2^31 (page_magic)
  int page_sh;
  int rope_w;
  int rms_off_b;  // byte offset of the rms tail inside a row
  const float* k_scale;
  float sm_scale, logit_cap;
  const int* bt;
  int64_t bt_stride;
  const int* seq_lens;
  int n_req;      // requests = rows / qrows
  int qrows, hpg; // verify tokens per request, heads per latent group
  int heads;      // heads per row (= groups * hpg)
  void* out;
  int64_t o_sr, o_sh;
  int out_dt;
  void* lse;
  int64_t lse_sr;
  int lse_dt;
  int num_splits, split_align;
  float* ws;
  int64_t ws_sr, ws_sh, ws_ss;
  // balanced mode
  int nwg;
  int* plan;        // [0] = chunk (tiles per workgroup), [1] = total tiles, [2 + b] = prefix C_b
  float* part_o;    // [(nwg + n_req), qrows*heads, Dv]
  float* part_lse;  // [(nwg + n_req), qrows*heads]
  int q_vec;        // query rows and strides 16-byte aligned: 16-byte query loads (else element loads)
  int hsplit;       // warp-specialized kernel: workgroups sharing a request's token range, each with
                    // heads/hsplit of its heads (balanced mode: nwg ranges x hsplit workgroups)
  uint32_t page_bound;  // block-table entries must lie in [0, page_bound)
  int* status;          // QMLA_ERR_PAGE is stored here when one does not (may be null)
  int plan_sw;          // plan tiles charged for a request switch (see plan_tiles): read by the
                        // combine and the plan kernel; the decode kernels have their family's as a
                        // constant
  int part_h;           // balanced partial outputs in fp16 and without the fp8 scale (fp8 caches:
                        // |value| <= 448), which the combine applies; else fp32
};

// x / d = (x * mul) >> sh for 0 <= x < 2^31, 1 <= d < 2^31: sh = 31 + ceil(log2 d), mul = ceil(2^sh / d) <
// 2^32. With e = mul * d - 2^sh < d <= 2^(sh - 31), x * mul / 2^sh = x/d + (x * e) / (d * 2^sh) lies less
// than 1/d above x/d, so both have the same integer part.
inline void page_magic(int d, uint32_t& mul, int& sh) {
  int l = 0;
  while (((int64_t)1 << l) < d) ++l;
  sh = 31 + l;
  mul = (uint32_t)((((uint64_t)1 << sh) + (uint64_t)d - 1) / (uint64_t)d);
}
__host__ __device__ __forceinline__ uint64_t magic_div(uint32_t x, uint32_t mul, int sh) { return ((uint64_t)x * mul) >> sh; }
__device__ __forceinline__ int page_div(const KParams& p, int x) { return (int)magic_div((uint32_t)x, p.page_mul, p.page_sh); }

// A block-table entry checked against the page bound: an entry outside [0, page_bound) reads page 0
// (in bounds) and raises `bad`, which the kernel reports once its memory traffic has drained.
__device__ __forceinline__ int checked_page(const KParams& p, int id, int& bad) {
  const bool ok = (uint32_t)id < p.page_bound;
  bad |= ok ? 0 : 1;
  return ok ? id : 0;
}
__device__ __forceinline__ void report_pages(const KParams& p, int bad) {
  if (bad && p.status) *p.status = QMLA_ERR_PAGE;
}

// 8 consecutive query elements: one 16-byte load when the caller's query rows are 16-byte aligned,
// else eight element loads (queries are read once per request or segment, so this costs nothing
// that shows). `vec` is the same for every lane.
__device__ __forceinline__ bf16x8 load_q8(const __bf16* ptr, bool vec) {
  if (vec) return *reinterpret_cast<const bf16x8*>(ptr);
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = ptr[e];
  return v;
}

__device__ __forceinline__ void store_out(void* base, int dt, int64_t idx, float v) {
  if (dt == QMLA_DT_BF16) reinterpret_cast<__bf16*>(base)[idx] = (__bf16)v;
  else if (dt == QMLA_DT_F16) reinterpret_cast<_Float16*>(base)[idx] = (_Float16)v;
  else reinterpret_cast<float*>(base)[idx] = v;
}

// Where the result of one token range goes.
struct SegOut {
  bool final_out;       // write normalized output + lse directly
  float* po;            // partial output base of this request (query-row 0 of it)
  int64_t po_sr, po_sh; // float strides for (verify token of the request, head)
  float* plse;          // balanced-mode lse base (nullptr: lse stored after the Dv columns)
  int64_t plse_sr;
};

// request length: the last flattened row of the request carries it (mla_impl.py:628-662)
__device__ __forceinline__ int req_len(const KParams& p, int req) {
  int L = p.seq_lens[(int64_t)req * p.qrows + p.qrows - 1];
  return L > 0 ? L : 0;
}

// ---- the balanced plan, computed by the decode kernels themselves ---------------------------------
// Request b owns plan tiles [C_b, C_b + T_b) of the concatenated requests, with T_b = ceil(L_b /
// PLAN_TILE) + plan_sw for a non-empty request (0 for an empty one) and C_b the exclusive prefix of
// the T's; workgroup w of nwg owns plan tiles [w*chunk, min((w+1)*chunk, total)) with chunk =
// ceil(total / nwg). A request's first plan_sw tiles hold no tokens: they charge the fixed work of
// a piece (the query load, the output write) to the workgroup that starts the request, so a
// workgroup holding two pieces gets fewer tokens than one holding one; the following tiles hold
// PLAN_TILE tokens each. Every workgroup derives
// its own range from seq_lens at its start (no planning launch: a launch of its own costs more
// than the scan, and inside a HIP graph far more), and workgroup 0 also stores the plan for the
// balanced combine.

// inclusive prefix sums over the 64 lanes, all of them active: DPP row shifts inside each 16 lanes,
// then the last lane of a row added to the rows after it
__device__ __forceinline__ int wave_incl_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);   // row_shr 1, 2, 4, 8
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);   // row_bcast 15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);   // row_bcast 31 into rows 2, 3
  return x;
}
__device__ __forceinline__ int lane_value(int x, int lane) { return __builtin_amdgcn_readlane(x, lane); }

template <int SW>
__device__ __forceinline__ int len_tiles(int L) {
  return L > 0 ? (L + PLAN_TILE - 1) / PLAN_TILE + SW : 0;
}
template <int SW>
__device__ __forceinline__ int plan_tiles(const KParams& p, int b) {
  return len_tiles<SW>(req_len(p, b));
}

// The tokens [a, e) of a request of length L with plan tiles [c0, c1) that plan tiles [lo, hi) hold
// (e <= a: none), and whether they are all of its tokens.
struct PieceTok {
  int a, e;
  bool whole;
};
template <int SW>
__device__ __forceinline__ PieceTok piece_tokens(int L, int c0, int c1, int lo, int hi) {
  const int v_lo = (lo > c0 ? lo : c0) - c0 - SW, v_hi = (hi < c1 ? hi : c1) - c0 - SW;
  const int t_lo = v_lo > 0 ? v_lo : 0, t_hi = v_hi > 0 ? v_hi : 0;
  PieceTok r;
  r.a = t_lo * PLAN_TILE;
  r.e = t_hi * PLAN_TILE < L ? t_hi * PLAN_TILE : L;
  r.whole = t_lo == 0 && t_hi == c1 - c0 - SW;
  return r;
}

struct BalRange {
  int lo, hi;      // plan tiles of this workgroup
  int chunk, total;
  int b0, c0;      // the last request with C_b <= lo, and its C_b
  int len[4];      // lane's lengths: request 64k + lane (0 past the last)
};

// One wave computes workgroup w's range (wave-uniform results; any wave may call it). The lengths of
// the first 256 requests are loaded at once and kept for the second pass; with a load and a scan over
// LDS permutes per 64 requests in each pass, range and window took 3.5 us at a workgroup's start, 2.4
// now, with the page divisions by multiplication (one request of 1300 tokens).
template <int SW>
__device__ inline BalRange balanced_range(const KParams& p, int w) {
  constexpr int NK = 4;
  const int lane = threadIdx.x & 63;
  BalRange r;
  r.chunk = 1;
  r.lo = r.hi = r.total = r.b0 = r.c0 = 0;
#pragma unroll
  for (int k = 0; k < NK; ++k) r.len[k] = 0;
  if (p.n_req <= 0) return r;
  int t[NK], incl[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int b = 64 * k + lane;
    t[k] = req_len(p, b < p.n_req ? b : p.n_req - 1);
  }
  int total = 0;
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    r.len[k] = 64 * k + lane < p.n_req ? t[k] : 0;
    t[k] = len_tiles<SW>(r.len[k]);
    incl[k] = wave_incl_sum(t[k]);
    total += lane_value(incl[k], 63);
  }
  for (int base = 64 * NK; base < p.n_req; base += 64) {
    const int b = base + lane;
    total += lane_value(wave_incl_sum(b < p.n_req ? plan_tiles<SW>(p, b) : 0), 63);
  }
  r.total = total;
  r.chunk = total > 0 ? (total + p.nwg - 1) / p.nwg : 1;
  r.lo = w * r.chunk;
  r.hi = r.lo + r.chunk < total ? r.lo + r.chunk : total;
  if (r.lo >= r.hi) return r;
  // the last request with C_b <= lo among 64 requests from base, whose tiles start at `run`
  auto find = [&](int base, int run, int tiles, int in) {
    const int c = run + in - tiles;
    const uint64_t m = __builtin_amdgcn_ballot_w64(base + lane < p.n_req && c <= r.lo);
    if (m) {
      const int x = 63 - __builtin_clzll(m);
      r.b0 = base + x;
      r.c0 = lane_value(c, x);
    }
  };
  int run = 0;
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    find(64 * k, run, t[k], incl[k]);
    run += lane_value(incl[k], 63);
  }
  for (int base = 64 * NK; base < p.n_req && run <= r.lo; base += 64) {
    const int b = base + lane;
    const int tb = b < p.n_req ? plan_tiles<SW>(p, b) : 0;
    const int in = wave_incl_sum(tb);
    find(base, run, tb, in);
    run += lane_value(in, 63);
  }
  return r;
}

// One wave of one workgroup stores the plan the balanced combine reads: [0] chunk, [1] total,
// [2 + b] = C_b for b <= n_req.
template <int SW>
__device__ inline void store_plan(const KParams& p) {
  const int lane = threadIdx.x & 63;
  int run = 0;
  for (int base = 0; base <= p.n_req; base += 64) {
    const int b = base + lane;
    const int t = b < p.n_req ? plan_tiles<SW>(p, b) : 0;
    const int incl = wave_incl_sum(t);
    if (b <= p.n_req) p.plan[2 + b] = run + incl - t;
    run += lane_value(incl, 63);
  }
  if (lane == 0) {
    p.plan[0] = run > 0 ? (run + p.nwg - 1) / p.nwg : 1;
    p.plan[1] = run;
  }
}

// Tokens per split in the fixed-split mode: ceil(ceil(L/S)/align)*align (mla_decode_attention.py:389-396).
__device__ __forceinline__ int split_len(const KParams& p, int L) {
  int per = (L + p.num_splits - 1) / p.num_splits;
  if (p.split_align > 0) per = (per + p.split_align - 1) / p.split_align * p.split_align;
  return per;
}

// Output of request b's token range in this workgroup: fixed splits write the reference's
// attn_logits row of split blockIdx.x; the balanced mode writes slot blockIdx.x + b of the partial
// buffers; final_out (the workgroup covers the whole request) writes the normalized output directly.
template <int DV>
__device__ __forceinline__ SegOut seg_out(const KParams& p, int b, bool final_out, int w = -1) {
  if (w < 0) w = blockIdx.x;   // the workgroup's split (fixed) or range (balanced)
  SegOut so;
  so.final_out = final_out;
  if (p.num_splits > 0) {
    so.po = p.ws + (int64_t)b * p.qrows * p.ws_sr + (int64_t)w * p.ws_ss;
    so.po_sr = p.ws_sr;
    so.po_sh = p.ws_sh;
    so.plse = nullptr;
    so.plse_sr = 0;
  } else {
    const int nrow = p.qrows * p.heads;
    const int64_t slot = (int64_t)w + b;
    so.po = p.part_o + slot * nrow * DV;
    so.po_sr = (int64_t)p.heads * DV;
    so.po_sh = DV;
    so.plse = p.part_lse + slot * nrow;
    so.plse_sr = p.heads;
  }
  return so;
}

// The rows of one finished piece: element (verify token j, head h, column c) of the output goes to
// base + (j*sr + h*sh + c) elements of dt, scaled by num / (row sum); its lse to
// lse + j*lse_sr + h*lse_sh elements of lse_dt (no lse when null).
struct RowOut {
  char* base;
  int dt;
  int64_t sr, sh;
  float num;
  char* lse;
  int lse_dt;
  int64_t lse_sr, lse_sh;
};
__device__ __forceinline__ int out_bytes(int dt) { return dt == QMLA_DT_F32 ? 4 : 2; }
// rows of the request whose first flattened row is row0, as `so` says: final output, balanced partial
// (fp16 without the fp8 scale, or fp32) or fixed-split partial (fp32, the lse after the DV columns)
template <int DV>
__device__ __forceinline__ RowOut row_out(const KParams& p, const SegOut& so, int row0, float kscale) {
  RowOut o;
  if (so.final_out) {
    o.dt = p.out_dt;
    o.base = reinterpret_cast<char*>(p.out) + (int64_t)row0 * p.o_sr * out_bytes(o.dt);
    o.sr = p.o_sr;
    o.sh = p.o_sh;
    o.num = kscale;   // fp8 values were accumulated unscaled
    o.lse_dt = p.lse_dt;
    o.lse = p.lse ? reinterpret_cast<char*>(p.lse) + (int64_t)row0 * p.lse_sr * out_bytes(o.lse_dt) : nullptr;
    o.lse_sr = p.lse_sr;
    o.lse_sh = 1;
  } else {
    const bool half = so.plse && p.part_h;
    o.dt = half ? QMLA_DT_F16 : QMLA_DT_F32;
    o.base = reinterpret_cast<char*>(so.po);
    o.sr = so.po_sr;
    o.sh = so.po_sh;
    o.num = half ? 1.0f : kscale;
    o.lse_dt = QMLA_DT_F32;
    o.lse = reinterpret_cast<char*>(so.plse ? so.plse : so.po + DV);
    o.lse_sr = so.plse ? so.plse_sr : so.po_sr;
    o.lse_sh = so.plse ? 1 : so.po_sh;
  }
  return o;
}

// 4 consecutive columns in one store; the caller's rows may be aligned to their elements only
typedef f32x4 f32x4_e __attribute__((aligned(4)));
typedef f16x4 f16x4_e __attribute__((aligned(2)));
typedef bf16x4 bf16x4_e __attribute__((aligned(2)));
template <int DT>
__device__ __forceinline__ void store_out4(char* ptr, const f32x4& v) {
  if constexpr (DT == QMLA_DT_F32) *reinterpret_cast<f32x4_e*>(ptr) = v;
  else if constexpr (DT == QMLA_DT_F16) *reinterpret_cast<f16x4_e*>(ptr) = f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
  else *reinterpret_cast<bf16x4_e*>(ptr) = bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
}

// Stores one row's columns from 16x16 accumulator tiles of O^T = V^T . P^T: lane (lg, n) holds columns
// 16cb + 4lg + i of row n, scaled by inv (num / the row's sum). e is the element offset of the row's
// first column, live false for rows past the request's. A tile's columns go out in one 8- or 16-byte
// store a lane and the output's type is branched on once. A finished request of two row blocks, by
// timestamps: 3.4 us with O = P . V (a lane holding column n of four rows: 64 stores of 2 or 4 bytes a lane
// in about 1000 basic blocks), 2.3 us with that transposed in registers before the store, 2.0 us as it is
// (0.35 for sums and addresses, 0.75 a row block).
template <int CB>
__device__ __forceinline__ void store_row(const RowOut& o, const f32x4 (&acc)[CB], float inv, int64_t e, bool live) {
  if (!live) return;
  const int c0 = 4 * ((threadIdx.x & 63) >> 4);
  auto put = [&](auto dtc) {
    constexpr int DT = decltype(dtc)::value, ES = DT == QMLA_DT_F32 ? 4 : 2;
    char* ptr = o.base + (e + c0) * ES;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) store_out4<DT>(ptr + 16 * ES * cb, acc[cb] * inv);
  };
  if (o.dt == QMLA_DT_F16) put(std::integral_constant<int, QMLA_DT_F16>{});
  else if (o.dt == QMLA_DT_F32) put(std::integral_constant<int, QMLA_DT_F32>{});
  else put(std::integral_constant<int, QMLA_DT_BF16>{});
}

// Calls f(req, a, e, L, so) for every token range [a, e) this workgroup owns.
//   fixed splits (num_splits > 0): grid (S, n_req); split s covers [s*per, min((s+1)*per, L)) with
//     per = ceil(ceil(L/S)/align)*align, as the reference's stage 1 (mla_decode_attention.py:389-396);
//     partials go to attn_logits [rows, heads, S, Dv+1].
//   balanced (num_splits == 0): workgroup w owns global PLAN_TILE-token tiles [w*chunk, (w+1)*chunk)
//     of the concatenated requests; a request it covers alone is finished in place, others leave a
//     partial in slot w + b.
template <int DV, int SW, class F>
__device__ __forceinline__ void for_each_segment(const KParams& p, F&& f) {
  // one call site of f, so the (large, inlined) segment body exists once per kernel
  const bool fixed = p.num_splits > 0;
  int b_lo, b_hi, lo = 0, hi = 0, c = 0;
  if (fixed) {
    b_lo = blockIdx.y;
    b_hi = b_lo + 1;
  } else {
    const BalRange r = balanced_range<SW>(p, blockIdx.x);
    lo = r.lo;
    hi = r.hi;
    if (lo >= hi) return;
    b_lo = r.b0;   // the request whose tiles contain lo (or an empty one right before it)
    c = r.c0;
    b_hi = p.n_req;
  }
  for (int b = b_lo; b < b_hi; ++b) {
    const int L = req_len(p, b);
    int a, e;
    SegOut so;
    if (fixed) {
      const int per = split_len(p, L);
      a = per * (int)blockIdx.x;
      e = a + per < L ? a + per : L;
      so = seg_out<DV>(p, b, p.num_splits == 1);
    } else {
      const int c0 = c, c1 = c + (L > 0 ? (L + PLAN_TILE - 1) / PLAN_TILE + SW : 0);
      c = c1;
      if (c0 >= hi) break;
      if (c1 <= lo) continue;
      const PieceTok pt = piece_tokens<SW>(L, c0, c1, lo, hi);
      a = pt.a;
      e = pt.e;
      so = seg_out<DV>(p, b, pt.whole);
    }
    if (e <= a) continue;
    f(b, a, e, L, so);
  }
}

// Cached rows on 16-byte boundaries (cache base, page stride and row stride): every kernel family
// stages them with 16-byte LDS-DMA loads. Rows on 4-byte boundaries only (the unpadded 12-head rows
// of the reference's numerics test) take the narrow-row instances, which stage 4 bytes per lane.
inline bool rows16(const qmla_decode_params* p) {
  const int eb = p->kv_dtype == QMLA_KV_FP8 ? 1 : 2;
  return ((uintptr_t)p->kv_cache & 15) == 0 && (p->page_stride * eb) % 16 == 0 && (p->token_stride * eb) % 16 == 0;
}

// ---- host-side interface of the warp-specialized translation unit (qmla_ws.hip) ----
int ws_select(const qmla_decode_params* p);
int ws_head_split(const qmla_decode_params* p);
int ws_launch(int inst, const qmla_decode_params* p, const KParams& k, int nwg, hipStream_t st);

// ---- host-side interface of the row-owner translation unit (qmla_ro.hip) ----
// Index of a compiled row-owner instance for these params (GLA-g2 on fp8 + log8 rows), or -1.
int ro_select(const qmla_decode_params* p);
int ro_launch(int inst, const qmla_decode_params* p, const KParams& k, int nwg, hipStream_t st);

// ---- host-side interface of the wide-row warp-specialized translation unit (qmla_wsb.hip) ----
// Index of a compiled instance for these params (bf16 rows, the deployed fp8 rows), or -1.
int wsb_select(const qmla_decode_params* p);
int wsb_launch(int inst, const qmla_decode_params* p, const KParams& k, int nwg, hipStream_t st);

// ---- host-side interface of the column-split translation unit (qmla_cs.hip) ----
// Index of a compiled column-split instance for these params, or -1.
int cs_select(const qmla_decode_params* p);
// Workgroups per token range (row splits along gridDim.z) of the selected instance, or 0.
int cs_row_splits(const qmla_decode_params* p);
// Launch the partial pass of column-split instance `inst` (grid per split mode).
int cs_launch(int inst, const qmla_decode_params* p, const KParams& k, int nwg, hipStream_t st);

}  // namespace qmla
