// qmla_write.hip -- gfx950 cache-row kernels: the writer (one new token per input row into its paged
// cache slot) and the prefill context gather (paged rows back into a dense bf16 workspace).
//
// Reference: qwen_mla/mla_impl.py:309-342 (QwenMLATritonImpl.do_kv_cache_update, the FP8 writer
// with log8 or bf16-byte rms tails) and vLLM's concat_and_cache_mla for the rows the plugin hands
// to it (bf16 caches; FP8 caches whose rms is e4m3). Up to a few thousand rows, and for bf16 caches,
// one wave per row: lane l converts latent elements [8l, 8l+8) (and further 512-column blocks for wider
// latents), lanes 0.. the rope in 8s and the rms tail one head each; more FP8 rows go two or four to a
// wave (write_rows_kernel, gather_rows_kernel).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qmla.h"
#include "qmla_common.h"
#include "qmla_device.h"

namespace qmla {
// token / page_size for tokens below 2^31 by multiplication (page_magic); mul 0: a 64-bit division
// (cache of 2^31 slots or more)
struct PageDiv {
  uint32_t mul;
  int sh, size;
};
static PageDiv page_div_of(int page_size, int64_t tokens) {
  PageDiv d{0u, 0, page_size};
  if (tokens <= 0x7fffffff) page_magic(page_size, d.mul, d.sh);
  return d;
}
__device__ __forceinline__ int64_t page_of(const PageDiv& d, int64_t tok) {
  return d.mul ? (int64_t)magic_div((uint32_t)tok, d.mul, d.sh) : tok / d.size;
}
// flat slots of a wave's rows: slot q of rows of n slots is slot (q - r n) of row r = q / n, from a
// 24-bit multiplication (q < 2^10, exact below 2^20 / n)
__device__ __forceinline__ uint32_t flat_mul(int n) { return ((1u << 20) + (uint32_t)n - 1) / (uint32_t)n; }
__device__ __forceinline__ int flat_row(int q, uint32_t mul) { return (int)(__umul24((uint32_t)q, mul) >> 20); }
__device__ __forceinline__ int64_t lane64(int64_t v, int lane) {   // another lane's value
  const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, lane), hi = (uint32_t)__shfl((int)(uint32_t)((uint64_t)v >> 32), lane);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ int64_t uniform64(int64_t v, int lane) {   // lane's value as a scalar
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), lane);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
// rows from which FP8 rows are written and gathered several to a wave. Writer, rank 512 / 768 / 1792:
// 2048 rows 3.1 / 3.4 / 4.2 us at one a wave, 3.3 / 3.5 / 4.5 at two; 3000 rows 3.5 / 4.0 / 5.0 and 3.6 /
// 4.1 / 5.3; 4096 rows 4.0 / 4.6 / 5.9 and 3.7 / 4.2 / 5.7. Gather: 4096 rows 4.8 / 5.2 / 7.4 and 4.5 /
// 5.4 / 7.9, 12001 rows 9.2 / 9.6 / 14.4 and 7.6 / 9.2 / 14.2
constexpr int kWriteRowsMin = 4096, kWriteRowsMin2 = 65536, kWriteWideMax = 131072;
constexpr int kGatherRowsMin = 4096;
namespace wr {

constexpr int ROWS_PER_WG = 4;

struct WParams {
  const uint16_t* kv_c;
  int64_t kv_c_stride;
  const uint16_t* k_pe;
  int64_t k_pe_stride;
  const int64_t* slots;
  int n, d_c, rope_w, rms_heads, kv_dtype, rms_mode;
  const float* k_scale;
  char* cache;
  int64_t page_stride, token_stride;
  PageDiv page;
  int64_t num_slots;
};

__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// clamp(x * inv, -448, 448) in fp32 (NaN stays NaN, as torch.clamp leaves it)
__device__ __forceinline__ float sat448(float x, float inv) {
  const float v = x * inv;
  return v > 448.0f ? 448.0f : (v < -448.0f ? -448.0f : v);
}

// four fp32 values -> four e4m3fn bytes, round to nearest even (v_cvt_pk_fp8_f32, OCP e4m3 on gfx950)
__device__ __forceinline__ uint32_t pack_e4m3(float a, float b, float c, float d) {
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
  return (uint32_t)w;
}

// 8 bf16 inputs -> 8 e4m3 bytes
__device__ __forceinline__ uint2 quant8r(const uint4 raw, float inv) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
  float f[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = sat448(bf16_to_f32((uint16_t)(w[i] & 0xFFFF)), inv);
    f[2 * i + 1] = sat448(bf16_to_f32((uint16_t)(w[i] >> 16)), inv);
  }
  return make_uint2(pack_e4m3(f[0], f[1], f[2], f[3]), pack_e4m3(f[4], f[5], f[6], f[7]));
}
__device__ __forceinline__ uint2 quant8(const uint16_t* src, float inv) {
  return quant8r(*reinterpret_cast<const uint4*>(src), inv);
}

// log8 code of one rms value: round-half-even((log2(max(r, 1e-30)) + 3) * (255 / 6)), clamped to
// [0, 255]; the logarithm is evaluated in double and rounded once to fp32, the rest in fp32
__device__ __forceinline__ uint32_t log8_code(float r) {
  const float rc = r < 1e-30f ? 1e-30f : r;   // clamp_min keeps NaN
  const float lg = (float)log2((double)rc);
  const float c = rintf((lg - (-3.0f)) * 42.5f);
  return (uint32_t)(c < 0.0f ? 0.0f : (c > 255.0f ? 255.0f : c));
}
// The same code from the hardware log2 (within 2 ulp of the rounded double one): (lg + 3) * 42.5
// then moves by less than 2e-4 inside the code range, so wherever it lies 1e-3 or more from a
// rounding midpoint it rounds as the double path does; the few values nearer one take that path.
__device__ __forceinline__ uint32_t log8_code_fast(float r) {
  const float rc = r < 1e-30f ? 1e-30f : r;
  const float y = (__builtin_amdgcn_logf(rc) - (-3.0f)) * 42.5f;
  if (fabsf(y - floorf(y) - 0.5f) < 1e-3f) return log8_code(r);
  const float c = rintf(y);
  return (uint32_t)(c < 0.0f ? 0.0f : (c > 255.0f ? 255.0f : c));
}

// One wave a row: bf16 caches, and FP8 rows outside write_rows_kernel's limits.
__global__ __launch_bounds__(64 * ROWS_PER_WG) void write_kernel(const WParams p) {
  const int lane = threadIdx.x & 63;
  const int row = (int)blockIdx.x * ROWS_PER_WG + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (row >= p.n) return;
  int64_t slot = p.slots[row];
  if (slot < 0) slot = 0;
  if (slot >= p.num_slots) return;
  const int64_t page = page_of(p.page, slot), tok = slot - page * p.page.size;
  char* dst = p.cache + page * p.page_stride + tok * p.token_stride;
  const uint16_t* kc = p.kv_c + (int64_t)row * p.kv_c_stride;
  const uint16_t* kp = p.k_pe + (int64_t)row * p.k_pe_stride;

  if (p.kv_dtype == QMLA_KV_FP8) {
    const float inv = 1.0f / *p.k_scale;
    for (int c = 8 * lane; c < p.d_c; c += 512)
      *reinterpret_cast<uint2*>(dst + c) = quant8(kc + c, inv);
    // the rope in 8-element groups, then the 1-7 elements before an rms tail that is not 8-aligned
    // one by one (the plugin's rope 116): a group must not spill into the tail other lanes write
    const int r8 = p.rope_w & ~7;
    for (int c = 8 * lane; c < r8; c += 512)
      *reinterpret_cast<uint2*>(dst + p.d_c + c) = quant8(kp + c, inv);
    if (lane < p.rope_w - r8) {
      const int c = r8 + lane;
      dst[p.d_c + c] = (char)(pack_e4m3(sat448(bf16_to_f32(kp[c]), inv), 0.f, 0.f, 0.f) & 0xFF);
    }
    char* rt = dst + p.d_c + p.rope_w;
    for (int h = lane; h < p.rms_heads; h += 64) {
      const uint16_t rb = kp[p.rope_w + h];
      if (p.rms_mode == QMLA_RMS_LOG8) {
        rt[h] = (char)log8_code_fast(bf16_to_f32(rb));
      } else if (p.rms_mode == QMLA_RMS_BF16_BYTES) {
        rt[2 * h] = (char)(rb & 0xFF);
        rt[2 * h + 1] = (char)(rb >> 8);
      } else if (p.rms_mode == QMLA_RMS_E4M3) {
        rt[h] = (char)(pack_e4m3(sat448(bf16_to_f32(rb), inv), 0.f, 0.f, 0.f) & 0xFF);
      }
    }
  } else {
    uint16_t* d16 = reinterpret_cast<uint16_t*>(dst);
    for (int c = 8 * lane; c < p.d_c; c += 512)
      *reinterpret_cast<uint4*>(d16 + c) = *reinterpret_cast<const uint4*>(kc + c);
    const int pe = p.rope_w + p.rms_heads;
    for (int c = lane; c < pe; c += 64) d16[p.d_c + c] = kp[c];
  }
}

// FP8 rows: one wave writes R rows. Whole 512-column blocks of a row go one 8-column chunk to a lane
// (row addresses in scalar registers); the chunks left over, the 1-7 rope elements before an rms tail
// that is not 8-aligned, and the rms elements of the R rows are each dealt out flat over the wave (the
// chunks in FP passes a row: up to 64 FP of them). Every load is in flight before the first conversion.
// The same bytes as write_kernel.
//
// What bounds it: below some 20000 rows the launch of the waves and each one's chain of slot, row and
// store, above that memory (65536 rows of rank 512: 118 MB in 23 us, 5.1 TB/s). 12001 rows of rank
// 512 / 768 / 1792 at one row a wave 7.2 / 9.3 / 14.6 us (write_kernel), two rows 6.5 / 8.3 / 14.0,
// four 6.4 / 8.6 / 16.5; 200000 rows of rank 512 and 768, one row 111 / 143, two 72 / 117, four 75 / 120.
// The chunks' passes and the rms elements' in loops of their own: 65536 rows of rank 768 36.2 -> 32.0.
template <int R, int NF, int FP>
__global__ __launch_bounds__(256) void write_rows_kernel(const WParams p) {
  const int lane = threadIdx.x & 63;
  const int r0 = ((int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) * R;
  if (r0 >= p.n) return;
  const int nr = p.n - r0 < R ? p.n - r0 : R;
  const int nch = p.d_c >> 3, nfull = nch >> 6, rem = nch & 63, nrp = p.rope_w >> 3, npre = p.rope_w & 7;
  const int ns = rem + nrp, heads = p.rms_heads;
  const uint32_t ms = ns > 0 ? flat_mul(ns) : 0u, mh = heads > 0 ? flat_mul(heads) : 0u;
  const uint16_t* kc = p.kv_c + (int64_t)r0 * p.kv_c_stride;
  const uint16_t* kp = p.k_pe + (int64_t)r0 * p.k_pe_stride;
  // ---- loads (rows past the end repeat the last row's) ----
  const int64_t slot0 = p.slots[r0 + (lane < nr ? lane : nr - 1)];
  const float inv = 1.0f / *p.k_scale;
  uint4 lat[R][NF], fl[R * FP];
  uint16_t rm[R], pre = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const uint16_t* row = kc + (int64_t)(i < nr ? i : nr - 1) * p.kv_c_stride;
#pragma unroll
    for (int k = 0; k < NF; ++k)
      if (k < nfull) lat[i][k] = *reinterpret_cast<const uint4*>(row + 8 * (lane + 64 * k));
  }
#pragma unroll
  for (int i = 0; i < R * FP; ++i) {
    const int q = lane + 64 * i;
    if (64 * i < R * ns && q < nr * ns) {
      const int r = flat_row(q, ms), c = q - r * ns;
      fl[i] = *reinterpret_cast<const uint4*>(c < rem ? kc + r * p.kv_c_stride + 512 * nfull + 8 * c
                                                     : kp + r * p.k_pe_stride + 8 * (c - rem));
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int q = lane + 64 * i;
    if (64 * i < R * heads && q < nr * heads) {
      const int r = flat_row(q, mh);
      rm[i] = kp[r * p.k_pe_stride + p.rope_w + q - r * heads];
    }
  }
  const int pr = npre > 0 ? lane / npre : R, pe = lane - pr * npre;   // this lane's pre-tail element
  if (pr < nr) pre = kp[pr * p.k_pe_stride + 8 * nrp + pe];
  // ---- lane r: byte offset of row r0 + r's slot, or -1 (nothing to write) ----
  const int64_t slot = slot0 < 0 ? 0 : slot0;
  int64_t off = -1;
  if (lane < nr && slot < p.num_slots) {
    const int64_t page = page_of(p.page, slot);
    off = page * p.page_stride + (slot - page * p.page.size) * p.token_stride;
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int64_t o = uniform64(off, i);
    if (o < 0) continue;
#pragma unroll
    for (int k = 0; k < NF; ++k)
      if (k < nfull) *reinterpret_cast<uint2*>(p.cache + o + 8 * (lane + 64 * k)) = quant8r(lat[i][k], inv);
  }
#pragma unroll
  for (int i = 0; i < R * FP; ++i) {
    const int q = lane + 64 * i;
    if (64 * i < R * ns) {   // wave-uniform
      const int r = q < nr * ns ? flat_row(q, ms) : 0;
      const int64_t o = lane64(off, r);
      const int c = q - r * ns;
      if (q < nr * ns && o >= 0)
        *reinterpret_cast<uint2*>(p.cache + o + 8 * (c < rem ? 64 * nfull + c : nch + c - rem)) = quant8r(fl[i], inv);
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int q = lane + 64 * i;
    if (64 * i < R * heads) {
      const int r = q < nr * heads ? flat_row(q, mh) : 0;
      const int64_t o = lane64(off, r);
      const int h = q - r * heads;
      if (q < nr * heads && o >= 0) {
        char* rt = p.cache + o + p.d_c + p.rope_w;
        if (p.rms_mode == QMLA_RMS_LOG8) {
          rt[h] = (char)log8_code_fast(bf16_to_f32(rm[i]));
        } else if (p.rms_mode == QMLA_RMS_BF16_BYTES) {
          rt[2 * h] = (char)(rm[i] & 0xFF);
          rt[2 * h + 1] = (char)(rm[i] >> 8);
        } else {
          rt[h] = (char)(pack_e4m3(sat448(bf16_to_f32(rm[i]), inv), 0.f, 0.f, 0.f) & 0xFF);
        }
      }
    }
  }
  if (npre > 0) {
    const int64_t o = lane64(off, pr < nr ? pr : 0);
    if (pr < nr && o >= 0)
      p.cache[o + p.d_c + 8 * nrp + pe] = (char)(pack_e4m3(sat448(bf16_to_f32(pre), inv), 0.f, 0.f, 0.f) & 0xFF);
  }
}

// 8-column chunks of a row past its whole 512-column blocks
static int flat_chunks(int d_c, int rope_w) { return (d_c / 8) % 64 + rope_w / 8; }

// Which FP8 rows write_rows_kernel takes: up to 64 flat chunks a row (one pass), up to 128 below 1024
// latent columns (two). Two passes pay once memory bounds the writer: d_c 448 with 128 rope columns, one
// row a wave and two, 12001 rows 7.2 and 7.3 us, 65536 rows 29.7 and 25.0, 262144 rows 149 and 105 (768
// with 264: 9.3 and 9.2, 36.3 and 35.3, 188 and 157; 256 with 512: 7.6 and 7.6, 30.5 and 28.6, 157 and
// 134). From 1280 columns on they do so up to 131072 rows only (896 with 512: 65536 rows 52.4 and 44.9,
// 131072 rows 114 and 118, 262144 rows 223 and 234). One pass: from 1408 columns on up to 131072 rows only
// (rank 1792 with 232: 65536 rows 79.0 at one row a wave and 78.7 at two, 131072 rows 151 and 155, 262144
// rows 292 and 309; 1536 with 128: 66.0 and 64.6, 135 and 138, 266 and 277; 1280 with 64: 262144 rows 231
// and 229).
static bool several_rows(const qmla_cache_write_params* p, int ns, int heads) {
  const bool two = ns > 64;
  if (p->d_c >= 2048 || ns > (p->d_c < 1024 ? 128 : 64) || heads > 64) return false;
  if (p->n >= kWriteWideMax && p->d_c + p->rope_w >= (two ? 1280 : 1408)) return false;
  return p->n >= (two ? kWriteRowsMin2 : kWriteRowsMin);
}

}  // namespace wr
}  // namespace qmla

extern "C" int qmla_cache_write(const qmla_cache_write_params* p, void* stream) {
  using namespace qmla;
  if (!p) return QMLA_ERR_NULL;
  if (p->n == 0) return QMLA_OK;
  if (!p->kv_c || !p->k_pe || !p->slots || !p->cache) return QMLA_ERR_NULL;
  if (p->n < 0 || p->d_c <= 0 || p->d_c % 8 || p->rope_w < 0 || p->rms_heads < 0 || p->page_size <= 0 ||
      p->num_slots <= 0 || p->kv_c_stride < p->d_c)
    return QMLA_ERR_SHAPE;
  const bool fp8 = p->kv_dtype == QMLA_KV_FP8;
  if (!fp8 && p->kv_dtype != QMLA_KV_BF16) return QMLA_ERR_MODE;
  const int rb = fp8 ? (p->rms_mode == QMLA_RMS_BF16_BYTES ? 2 : (p->rms_mode == QMLA_RMS_NONE ? 0 : 1))
                     : (p->rms_mode == QMLA_RMS_BF16 ? 2 : 0);
  if (fp8 && p->rms_mode != QMLA_RMS_LOG8 && p->rms_mode != QMLA_RMS_BF16_BYTES && p->rms_mode != QMLA_RMS_E4M3 &&
      p->rms_mode != QMLA_RMS_NONE)
    return QMLA_ERR_MODE;
  if (!fp8 && p->rms_mode != QMLA_RMS_BF16 && p->rms_mode != QMLA_RMS_NONE) return QMLA_ERR_MODE;
  if (fp8 && !p->k_scale) return QMLA_ERR_NULL;
  const int pe_elems = p->rope_w + (rb ? p->rms_heads : 0);
  if (p->k_pe_stride < pe_elems) return QMLA_ERR_SHAPE;
  // the written bytes must fit one token slot
  const int64_t row_bytes = fp8 ? (int64_t)p->d_c + p->rope_w + (int64_t)rb * p->rms_heads
                                : 2 * ((int64_t)p->d_c + p->rope_w + (rb ? p->rms_heads : 0));
  if (row_bytes > p->token_stride || p->page_stride < p->token_stride * p->page_size) return QMLA_ERR_SHAPE;
  // 16-byte vector loads of kv_c and k_pe rows, 8- or 16-byte stores into the row
  if (((uintptr_t)p->kv_c | (uintptr_t)p->k_pe | (uintptr_t)p->cache) % 16 ||
      (p->kv_c_stride * 2) % 16 || (fp8 && (p->k_pe_stride * 2) % 16) || p->token_stride % 16 || p->page_stride % 16)
    return QMLA_ERR_ALIGN;
  wr::WParams k;
  k.kv_c = static_cast<const uint16_t*>(p->kv_c);
  k.kv_c_stride = p->kv_c_stride;
  k.k_pe = static_cast<const uint16_t*>(p->k_pe);
  k.k_pe_stride = p->k_pe_stride;
  k.slots = p->slots;
  k.n = p->n;
  k.d_c = p->d_c;
  k.rope_w = p->rope_w;
  k.rms_heads = rb ? p->rms_heads : 0;   // without rms elements k_pe rows may end after the rope
  k.kv_dtype = p->kv_dtype;
  k.rms_mode = p->rms_mode;
  k.k_scale = p->k_scale;
  k.cache = static_cast<char*>(p->cache);
  k.page_stride = p->page_stride;
  k.token_stride = p->token_stride;
  k.page = page_div_of(p->page_size, p->num_slots);
  k.num_slots = p->num_slots;
  void* args[] = {&k};
  const int ns = wr::flat_chunks(p->d_c, p->rope_w);
  if (fp8 && wr::several_rows(p, ns, k.rms_heads)) {
    constexpr int R = 2;
    const unsigned grid = (unsigned)((p->n + 4 * R - 1) / (4 * R));
    const void* fn = p->d_c >= 1024 ? (const void*)wr::write_rows_kernel<R, 3, 1>
                     : ns > 64      ? (const void*)wr::write_rows_kernel<R, 1, 2>
                                    : (const void*)wr::write_rows_kernel<R, 1, 1>;
    const hipError_t e = hipLaunchKernel(fn, dim3(grid), dim3(256), args, 0, (hipStream_t)stream);
    return e == hipSuccess ? QMLA_OK : QMLA_ERR_LAUNCH;
  }
  const unsigned grid = (unsigned)((p->n + wr::ROWS_PER_WG - 1) / wr::ROWS_PER_WG);
  const hipError_t e = hipLaunchKernel((const void*)wr::write_kernel, dim3(grid), dim3(64 * wr::ROWS_PER_WG), args,
                                       0, (hipStream_t)stream);
  return e == hipSuccess ? QMLA_OK : QMLA_ERR_LAUNCH;
}

// ---- prefill context gather (qwen_mla/ops/mla_gather.py:28-76) -----------------------------------
// One wave per destination row: the row's sequence, token and page from the chunk metadata, then the
// cached row copied (bf16 caches) or dequantized into the destination dtype (FP8 caches).
namespace qmla {
namespace ga {

constexpr int ROWS_PER_WG = 4;

struct GParams {
  const char* cache;
  int64_t page_stride, token_stride;
  PageDiv page;
  int num_pages, kv_dtype, rms_mode, rms_offset, rms_heads, row_elems;
  const float* scale;
  const int32_t* block_table;
  int64_t bt_stride;
  int num_seqs, bt_cols;
  const int32_t* cu_seq_lens;
  const int32_t* token_to_seq;
  const int32_t* seq_starts;
  int num_tokens;
  char* dst;
  int64_t dst_stride;
  int dst_dtype;
};

// one e4m3 byte (byte k of w) -> fp32; the conversion returns +0 for the negative zero 0x80, so the
// sign bit is put back (torch decodes 0x80 as -0.0, which survives the scale and the rounding)
__device__ __forceinline__ float e4m3_f32(int w, int k) {
  float f;
  switch (k) {
    case 0: f = __builtin_amdgcn_cvt_f32_fp8(w, 0); break;
    case 1: f = __builtin_amdgcn_cvt_f32_fp8(w, 1); break;
    case 2: f = __builtin_amdgcn_cvt_f32_fp8(w, 2); break;
    default: f = __builtin_amdgcn_cvt_f32_fp8(w, 3); break;
  }
  return __uint_as_float(__float_as_uint(f) | (((uint32_t)w >> (8 * k + 7)) & 1u) << 31);
}

// fp32 -> the destination dtype, round to nearest even; the sign bit is carried over explicitly so a
// negative zero stays negative whatever instruction the conversion compiles to
__device__ __forceinline__ uint16_t to_out(float x, int dt) {
  const uint16_t sign = (uint16_t)((__float_as_uint(x) >> 16) & 0x8000u);
  if (dt == QMLA_DT_F16) return (uint16_t)(__builtin_bit_cast(uint16_t, (_Float16)x) | sign);
  return (uint16_t)(__builtin_bit_cast(uint16_t, (__bf16)x) | sign);
}

// log8 code -> 2^(-3 + code * 6/255), rounded once from double
struct Log8Table {
  float v[256];
};
constexpr Log8Table make_log8() {
  Log8Table t{};
  for (int c = 0; c < 256; ++c) {
    const double x = -3.0 + c * (6.0 / 255.0);
    const int n = (int)(x + 8.0) - 8;                          // floor
    const double f = (x - n) * 0.693147180559945309417232121458;
    double term = 1.0, sum = 1.0;                              // e^f, 0 <= f < ln 2
    for (int k = 1; k < 28; ++k) {
      term *= f / k;
      sum += term;
    }
    t.v[c] = (float)(n >= 0 ? sum * (double)(1 << n) : sum / (double)(1 << -n));
  }
  return t;
}
__constant__ Log8Table kLog8 = make_log8();

// byte offset in the cache of destination row j, or -1 (nothing to write)
__device__ __forceinline__ int64_t row_offset(const GParams& p, int j) {
  const int s = p.token_to_seq[j];
  if (s < 0 || s >= p.num_seqs) return -1;
  int64_t tok = (int64_t)j - p.cu_seq_lens[s];
  if (p.seq_starts) tok += p.seq_starts[s];
  if (tok < 0 || tok >= (int64_t)p.bt_cols * p.page.size) return -1;
  const int64_t pi = page_of(p.page, tok);
  const int blk = p.block_table[(int64_t)s * p.bt_stride + pi];
  if (blk < 0 || blk >= p.num_pages) return -1;
  return (int64_t)blk * p.page_stride + (tok - pi * p.page.size) * p.token_stride;
}

// One wave a row: bf16 caches, and FP8 rows outside gather_rows_kernel's limits.
__global__ __launch_bounds__(64 * ROWS_PER_WG) void gather_kernel(const GParams p) {
  const int lane = threadIdx.x & 63;
  const int j = (int)blockIdx.x * ROWS_PER_WG + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (j >= p.num_tokens) return;
  const int64_t off = row_offset(p, j);
  if (off < 0) return;
  const char* row = p.cache + off;
  uint16_t* out = reinterpret_cast<uint16_t*>(p.dst) + (int64_t)j * p.dst_stride;

  if (p.kv_dtype == QMLA_KV_BF16) {
    const uint16_t* src = reinterpret_cast<const uint16_t*>(row);
    if (p.dst_dtype == QMLA_DT_BF16) {
      const int nv = p.row_elems / 8;
      for (int c = lane; c < nv; c += 64)
        reinterpret_cast<uint4*>(out)[c] = reinterpret_cast<const uint4*>(src)[c];
      for (int c = 8 * nv + lane; c < p.row_elems; c += 64) out[c] = src[c];
    } else {
      for (int c = lane; c < p.row_elems; c += 64) out[c] = to_out(__uint_as_float((uint32_t)src[c] << 16), p.dst_dtype);
    }
    return;
  }
  const float sc = *p.scale;
  // latent + rope: e4m3 * scale in fp32, rounded to the destination dtype; whole 8-byte groups as
  // vectors, the 1-7 bytes before an rms tail that is not 8-aligned one by one (the plugin's 12-head
  // rope-116 rows put the tail at 4 mod 8)
  const int c8 = p.rms_offset & ~7;
  for (int c = 8 * lane; c < c8; c += 512) {
    const uint2 raw = *reinterpret_cast<const uint2*>(row + c);
    const uint32_t w[2] = {raw.x, raw.y};
    uint32_t o[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int wv = (int)w[h];
      const float f0 = e4m3_f32(wv, 0) * sc, f1 = e4m3_f32(wv, 1) * sc;
      const float f2 = e4m3_f32(wv, 2) * sc, f3 = e4m3_f32(wv, 3) * sc;
      o[2 * h] = (uint32_t)to_out(f0, p.dst_dtype) | ((uint32_t)to_out(f1, p.dst_dtype) << 16);
      o[2 * h + 1] = (uint32_t)to_out(f2, p.dst_dtype) | ((uint32_t)to_out(f3, p.dst_dtype) << 16);
    }
    *reinterpret_cast<uint4*>(out + c) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  if (lane < p.rms_offset - c8) {
    const int c = c8 + lane;
    out[c] = to_out(e4m3_f32((int)(unsigned char)row[c], 0) * sc, p.dst_dtype);
  }
  // the rms tail: one element per head at rms_offset
  const unsigned char* tail = reinterpret_cast<const unsigned char*>(row) + p.rms_offset;
  for (int h = lane; h < p.rms_heads; h += 64) {
    float v;
    if (p.rms_mode == QMLA_RMS_LOG8) {
      v = kLog8.v[tail[h]];
    } else if (p.rms_mode == QMLA_RMS_BF16_BYTES) {
      const uint32_t bits = (uint32_t)tail[2 * h] | ((uint32_t)tail[2 * h + 1] << 8);
      if (p.dst_dtype == QMLA_DT_BF16) {
        out[p.rms_offset + h] = (uint16_t)bits;
        continue;
      }
      v = __uint_as_float(bits << 16);
    } else {
      v = e4m3_f32((int)tail[h], 0) * sc;
    }
    out[p.rms_offset + h] = to_out(v, p.dst_dtype);
  }
}

// 8 e4m3 bytes -> scaled, in the destination dtype
template <int DT>
__device__ __forceinline__ uint4 dequant8(const uint2 raw, float sc) {
  const uint32_t w[2] = {raw.x, raw.y};
  uint32_t o[4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int wv = (int)w[h];
    const float f0 = e4m3_f32(wv, 0) * sc, f1 = e4m3_f32(wv, 1) * sc;
    const float f2 = e4m3_f32(wv, 2) * sc, f3 = e4m3_f32(wv, 3) * sc;
    o[2 * h] = (uint32_t)to_out(f0, DT) | ((uint32_t)to_out(f1, DT) << 16);
    o[2 * h + 1] = (uint32_t)to_out(f2, DT) | ((uint32_t)to_out(f3, DT) << 16);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// FP8 rows: one wave gathers R destination rows. Lanes 0 .. R-1 resolve the rows' sequence, token and
// page together. Whole 512-byte blocks of a row go one 8-byte chunk to a lane (row addresses in scalar
// registers); the chunks left over, the 1-7 bytes before an rms tail that is not 8-aligned, and the
// rms elements of the R rows are each dealt out flat over the wave. Every load is in flight before the
// first conversion. The same values as gather_kernel.
//
// What bounds it: as write_rows_kernel, the waves and their chain (sequence, page, row) below some 20000
// rows, memory above. 16384 rows of rank 512 / 768 / 1792: 11.4 / 12.6 / 18.7 us at one row a wave
// (gather_kernel), 9.3 / 12.3 / 18.1 at two rows, 9.3 / 13.1 / 20.6 at four; 65536 rows 34.8 / 35.9 /
// 59.6 at one, 26.5 / 35.1 / 62.2 at two, 24.2 / 34.9 / 65.7 at four.
template <int DT, int R, int NF>
__global__ __launch_bounds__(256) void gather_rows_kernel(const GParams p) {
  const int lane = threadIdx.x & 63;
  const int j0 = ((int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) * R;
  if (j0 >= p.num_tokens) return;
  const int nr = p.num_tokens - j0 < R ? p.num_tokens - j0 : R;
  const int64_t off = lane < nr ? row_offset(p, j0 + lane) : -1;
  const int nch = p.rms_offset >> 3, npre = p.rms_offset & 7, nfull = nch >> 6, ns = nch & 63, heads = p.rms_heads;
  const uint32_t ms = ns > 0 ? flat_mul(ns) : 0u, mh = heads > 0 ? flat_mul(heads) : 0u;
  const float sc = *p.scale;
  uint16_t* out0 = reinterpret_cast<uint16_t*>(p.dst) + (int64_t)j0 * p.dst_stride;
  // ---- loads ----
  uint2 blk[R][NF], fl[R];
  uint32_t tb[R], pre = 0u;
  uint32_t flive = 0u, tlive = 0u;   // bit i: this lane's slot of pass i belongs to a row to write
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int64_t o = uniform64(off, i);
    if (o < 0) continue;
#pragma unroll
    for (int k = 0; k < NF; ++k)
      if (k < nfull) blk[i][k] = *reinterpret_cast<const uint2*>(p.cache + o + 8 * (lane + 64 * k));
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int q = lane + 64 * i;
    if (64 * i < R * ns) {   // wave-uniform
      const int r = q < nr * ns ? flat_row(q, ms) : 0;
      const int64_t o = lane64(off, r);
      if (q < nr * ns && o >= 0) {
        flive |= 1u << i;
        fl[i] = *reinterpret_cast<const uint2*>(p.cache + o + 512 * nfull + 8 * (q - r * ns));
      }
    }
    if (64 * i < R * heads) {
      const int r = q < nr * heads ? flat_row(q, mh) : 0;
      const int64_t o = lane64(off, r);
      if (q < nr * heads && o >= 0) {
        tlive |= 1u << i;
        const unsigned char* tail = reinterpret_cast<const unsigned char*>(p.cache + o) + p.rms_offset;
        const int h = q - r * heads;
        tb[i] = p.rms_mode == QMLA_RMS_BF16_BYTES ? ((uint32_t)tail[2 * h] | ((uint32_t)tail[2 * h + 1] << 8))
                                                  : (uint32_t)tail[h];
      }
    }
  }
  const int pr = npre > 0 ? lane / npre : R, pe = lane - pr * npre;   // this lane's pre-tail byte
  bool plive = false;
  if (npre > 0) {
    const int64_t o = lane64(off, pr < nr ? pr : 0);
    plive = pr < nr && o >= 0;
    if (plive) pre = (uint32_t)(unsigned char)p.cache[o + 8 * nch + pe];
  }
  // ---- conversions and stores ----
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (uniform64(off, i) < 0) continue;
    uint16_t* out = out0 + i * p.dst_stride;
#pragma unroll
    for (int k = 0; k < NF; ++k)
      if (k < nfull) *reinterpret_cast<uint4*>(out + 8 * (lane + 64 * k)) = dequant8<DT>(blk[i][k], sc);
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int q = lane + 64 * i;
    if (flive & (1u << i)) {
      const int r = flat_row(q, ms);
      *reinterpret_cast<uint4*>(out0 + r * p.dst_stride + 512 * nfull + 8 * (q - r * ns)) = dequant8<DT>(fl[i], sc);
    }
    if (tlive & (1u << i)) {
      const int r = flat_row(q, mh);
      uint16_t* out = out0 + r * p.dst_stride + p.rms_offset + q - r * heads;
      if (p.rms_mode == QMLA_RMS_LOG8) *out = to_out(kLog8.v[tb[i]], DT);
      else if (p.rms_mode == QMLA_RMS_E4M3) *out = to_out(e4m3_f32((int)tb[i], 0) * sc, DT);
      else *out = DT == QMLA_DT_BF16 ? (uint16_t)tb[i] : to_out(__uint_as_float(tb[i] << 16), DT);
    }
  }
  if (plive) out0[pr * p.dst_stride + 8 * nch + pe] = to_out(e4m3_f32((int)pre, 0) * sc, DT);
}

// Rows a wave of gather_rows_kernel, two or four. Below 1024 columns four pay from 16384 rows on where the
// rows' flat chunks then fit fewer passes each (576 columns 65536 rows 26.5 us at two and 24.2 at four; 884:
// 16384 rows 12.4 and 11.7, 65536 rows 35.3 and 31.6), and from 32768 rows on where they do not (1000
// columns, 61 chunks: 16384 rows 12.3 and 13.0, 30000 rows 18.5 and 19.4, 65536 rows 35.1 and 34.9, 200000
// rows 120 and 105; 704 columns: 30000 rows 15.5 and 16.2, 200000 rows 79 and 75). Up to 1280 columns four
// pay once the rows and their copies outgrow the memory-side cache (1024 columns: 131072 rows 63.7 and
// 66.2, 160000 rows 88 and 81, 262144 rows 157 and 138), and never at rank 1792 (200000 rows 209 and 232).
static int rows_per_wave(const qmla_gather_params* p) {
  const int n = p->num_tokens, ns = p->rms_offset / 8 % 64;
  if (p->rms_offset >= 1024) return p->rms_offset <= 1280 && n >= 150000 ? 4 : 2;
  const bool fewer = (4 * ns + 63) / 64 < 2 * ((2 * ns + 63) / 64);
  return n >= (fewer ? 16384 : 32768) ? 4 : 2;
}

}  // namespace ga
}  // namespace qmla

extern "C" int qmla_gather(const qmla_gather_params* p, void* stream) {
  using namespace qmla;
  if (!p) return QMLA_ERR_NULL;
  if (p->num_tokens == 0) return QMLA_OK;
  if (!p->cache || !p->block_table || !p->cu_seq_lens || !p->token_to_seq || !p->dst) return QMLA_ERR_NULL;
  if (p->num_tokens < 0 || p->page_size <= 0 || p->num_pages <= 0 || p->num_seqs <= 0 || p->bt_cols <= 0 ||
      p->bt_stride < p->bt_cols)
    return QMLA_ERR_SHAPE;
  if (p->dst_dtype != QMLA_DT_BF16 && p->dst_dtype != QMLA_DT_F16) return QMLA_ERR_MODE;
  const bool fp8 = p->kv_dtype == QMLA_KV_FP8;
  if (!fp8 && p->kv_dtype != QMLA_KV_BF16) return QMLA_ERR_MODE;
  int64_t width;
  if (fp8) {
    if (p->rms_mode != QMLA_RMS_LOG8 && p->rms_mode != QMLA_RMS_BF16_BYTES && p->rms_mode != QMLA_RMS_E4M3)
      return QMLA_ERR_MODE;
    if (!p->scale) return QMLA_ERR_NULL;
    if (p->rms_offset <= 0 || p->rms_heads < 0) return QMLA_ERR_SHAPE;
    const int64_t rb = p->rms_mode == QMLA_RMS_BF16_BYTES ? 2 : 1;
    if (p->rms_offset + rb * p->rms_heads > p->token_stride) return QMLA_ERR_SHAPE;
    width = (int64_t)p->rms_offset + p->rms_heads;
  } else {
    if (p->row_elems <= 0 || 2 * (int64_t)p->row_elems > p->token_stride) return QMLA_ERR_SHAPE;
    width = p->row_elems;
  }
  if (p->dst_stride < width || p->page_stride < p->token_stride * p->page_size) return QMLA_ERR_SHAPE;
  if (((uintptr_t)p->cache | (uintptr_t)p->dst) % 16 || p->token_stride % 16 || p->page_stride % 16 ||
      (p->dst_stride * 2) % 16)
    return QMLA_ERR_ALIGN;
  ga::GParams k;
  k.cache = static_cast<const char*>(p->cache);
  k.page_stride = p->page_stride;
  k.token_stride = p->token_stride;
  k.page = page_div_of(p->page_size, (int64_t)p->bt_cols * p->page_size);
  k.num_pages = p->num_pages;
  k.kv_dtype = p->kv_dtype;
  k.rms_mode = p->rms_mode;
  k.rms_offset = p->rms_offset;
  k.rms_heads = p->rms_heads;
  k.row_elems = p->row_elems;
  k.scale = p->scale;
  k.block_table = p->block_table;
  k.bt_stride = p->bt_stride;
  k.num_seqs = p->num_seqs;
  k.bt_cols = p->bt_cols;
  k.cu_seq_lens = p->cu_seq_lens;
  k.token_to_seq = p->token_to_seq;
  k.seq_starts = p->seq_starts;
  k.num_tokens = p->num_tokens;
  k.dst = static_cast<char*>(p->dst);
  k.dst_stride = p->dst_stride;
  k.dst_dtype = p->dst_dtype;
  void* args[] = {&k};
  if (fp8 && p->num_tokens >= kGatherRowsMin && p->rms_offset < 2048 && p->rms_heads <= 64) {
    const bool wide = p->rms_offset >= 1024, f16 = p->dst_dtype == QMLA_DT_F16;
    const int R = ga::rows_per_wave(p);
    const unsigned grid = (unsigned)((p->num_tokens + 4 * R - 1) / (4 * R));
#define QMLA_GA(RR, NF) \
    (f16 ? (const void*)ga::gather_rows_kernel<QMLA_DT_F16, RR, NF> : (const void*)ga::gather_rows_kernel<QMLA_DT_BF16, RR, NF>)
    const void* fn = wide ? (R == 2 ? QMLA_GA(2, 3) : QMLA_GA(4, 3)) : R == 2 ? QMLA_GA(2, 1) : QMLA_GA(4, 1);
#undef QMLA_GA
    const hipError_t e = hipLaunchKernel(fn, dim3(grid), dim3(256), args, 0, (hipStream_t)stream);
    return e == hipSuccess ? QMLA_OK : QMLA_ERR_LAUNCH;
  }
  const unsigned grid = (unsigned)((p->num_tokens + ga::ROWS_PER_WG - 1) / ga::ROWS_PER_WG);
  const hipError_t e = hipLaunchKernel((const void*)ga::gather_kernel, dim3(grid), dim3(64 * ga::ROWS_PER_WG), args,
                                       0, (hipStream_t)stream);
  return e == hipSuccess ? QMLA_OK : QMLA_ERR_LAUNCH;
}
