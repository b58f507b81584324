// pa_device.h - device code shared by the decode kernels (pa_decode.hip,
// pa_range.hip): argument block, streamed row loads, device-scope partials
// and their fold, element formats, wave-wide integer helpers and the
// sequence table.
#ifndef PA_DEVICE_H_
#define PA_DEVICE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pad {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u3_t __attribute__((ext_vector_type(3)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

constexpr float kNegInf = -__builtin_inff();
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kBlockTokens = 16;  // tokens per wave iteration (one MFMA tile)
constexpr int kMaxWaves = 8;
// Fewest 16-token blocks per split (or planned item): each workgroup's fixed
// costs (q load, wave merge, partial publish) stay small against its streaming.
constexpr int kMinBlocks = 16;
// Fewest blocks per split for short latency-bound sequences (split counts up
// to 16, which one merge round trip covers).
constexpr int kMinBlocksShort = 4;
// Units with more splits than this merge in two levels (groups of 16).
constexpr int kTwoLevelSplits = 48;
// A unit's workgroups fold its splits together from this many (split, row, 4
// columns) elements on (256 KB of partials), and up to kTwoLevelSplits splits
// (or 64 of the largest partials, 16 rows of 256): they wait on one line, one
// arrival after the other (us alone / shared: 2 x 16384 of 16/1 at 256, 64
// splits, 25.0 / 19.4; 2 x 32768 at 128, 64 splits, 16.8 / 17.3; 1 x 65536,
// 128 splits, 17.2 / 20.3).  With half the partials it gains nothing (8 x 8192
// of 16/1 at 128, 14.8 / 15.5).
constexpr int kSharedFoldElements = 16384;

// LDS of one workgroup (wave merge + MFMA staging) is capped so that the
// widest rows (head_dim 256, 16-row groups) still get 4 waves in a
// workgroup that fits a CU's 160 KB: one 2-wave workgroup per split left
// those shapes latency-bound (16/1 d256 batch 8 x 8192: 35.2 against
// 24.7 us).
constexpr int kLdsBudget = 136 * 1024;
// Headroom (base-2 units) a score may exceed the running reference max before
// the accumulators are rescaled; fp16 weights stay <= 2^8.
constexpr float kRescaleSlack = 8.0f;

// Largest batch the in-kernel work planner handles (4 sequences per lane).
constexpr int kPlanMaxBatch = 256;

struct Phase1Args {
  // Control fields first: they are read at the start of every workgroup.
  int gqa, ps, pps, num_splits, hkv, max_pages, batch;
  int nw;          // waves per workgroup (blockDim.x / 64)
  int ps_shift;    // log2(ps) when ps is a power of two, else -1
  int csr;         // 1: page ids from (indptr, indices, last_page_len)
  int balance;     // 1: items planned from the sequence lengths in-kernel;
                   // 2-4: the same on an oversubscribed grid (balance - 1
                   //    static splits per unit, pps pages each, on the
                   //    first workgroups when every sequence is full)
  int min_chunk;   // planner: fewest pages per item
  int pair_heads;  // 1: workgroups 8 apart take kv heads 2m and 2m+1 (see grid_pos)
  int wl_key;      // key of the launch's plan, matched against the work list's header
  float scale_log2;
  float v_fix;     // fp8 caches: V's scale, applied to the output rows
  int fold_polls;  // > 0: a unit's workgroups share the fold of its splits, each waiting at most this many polls
  const int32_t* bt;      // dense: block_table [B, max_pages]; CSR: indices
  const int32_t* sl;      // dense: seq_lens [B]
  const int32_t* indptr;  // CSR: [B + 1] offsets of each sequence's page ids in bt
  const int32_t* lpl;     // CSR: [B] tokens in each sequence's last page
  const int32_t* worklist;  // precomputed work items (header + one record per workgroup) or nullptr
  int64_t sbb, sbp;
  int64_t ssl;
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  _Float16* out;
  float* o_part;   // [G, gqa, D], one slot per workgroup of the grid
  float2* ml_part; // [G, gqa]  (m in base-2 units, l)
  int* counters;   // [B, Hkv] arrival counts, then per-slot group counts; zero between launches
  int64_t sqb, sqh;
  int64_t skp, sks, skh;
  int64_t svp, svs, svh;
  int64_t sob, soh;
  int64_t num_pages;
#ifdef PAD_TIMELINE
  int tl_launch;   // ring slot of this launch's stamps
#endif
};

// Token -> page index, and pages covering n tokens (shift for power-of-two
// page sizes).
__device__ __forceinline__ int page_of(const Phase1Args& a, int t) {
  return a.ps_shift >= 0 ? (t >> a.ps_shift) : t / a.ps;
}
// (n + ps - 1 can pass 2^31 where a length lies far beyond its table: unsigned.)
__device__ __forceinline__ int pages_for(const Phase1Args& a, int n) {
  const uint32_t t = (uint32_t)n + (uint32_t)a.ps - 1u;
  return (int)(a.ps_shift >= 0 ? t >> a.ps_shift : t / (uint32_t)a.ps);
}
// 16-token block -> page index (page_size a multiple of 16).
__device__ __forceinline__ int block_page(const Phase1Args& a, int jb) {
  return a.ps_shift >= 4 ? (jb >> (a.ps_shift - 4)) : jb / (a.ps / 16);
}

__device__ __forceinline__ float exp2_fast(float x) {
  return __builtin_amdgcn_exp2f(x);  // v_exp_f32; exp2(-inf) = 0
}

__device__ __forceinline__ float shfl_xor_f(float x, int m) {
  return __shfl_xor(x, m, 64);
}

// Sum over the 16 lanes of a DPP row (lanes 16r .. 16r+15), result in all.
__device__ __forceinline__ float row16_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xF, 0xF, false));   // quad_perm [2,3,0,1]
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xF, 0xF, false));  // row_half_mirror
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x140, 0xF, 0xF, false));  // row_mirror
  return x;
}

// NDW dwords (2*NDW halves) loaded from a 4*NDW-byte aligned address.
template <int NDW>
struct HVec {
  uint32_t w[NDW];
  __device__ __forceinline__ _Float16 h(int i) const {
    const uint32_t x = w[i >> 1];
    const uint16_t bits = (i & 1) ? (uint16_t)(x >> 16) : (uint16_t)(x & 0xffffu);
    return __builtin_bit_cast(_Float16, bits);
  }
  __device__ __forceinline__ h2_t h2(int i) const { return __builtin_bit_cast(h2_t, w[i]); }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < NDW; ++i) w[i] = 0u;
  }
};

template <int NDW>
__device__ __forceinline__ HVec<NDW> load_hvec(const _Float16* p) {
  HVec<NDW> r;
  if constexpr (NDW % 4 == 0) {
    const uint4* src = reinterpret_cast<const uint4*>(p);
#pragma unroll
    for (int i = 0; i < NDW / 4; ++i) {
      const uint4 x = src[i];
      r.w[4 * i + 0] = x.x; r.w[4 * i + 1] = x.y; r.w[4 * i + 2] = x.z; r.w[4 * i + 3] = x.w;
    }
  } else if constexpr (NDW % 2 == 0) {
    const uint2* src = reinterpret_cast<const uint2*>(p);
#pragma unroll
    for (int i = 0; i < NDW / 2; ++i) {
      const uint2 x = src[i];
      r.w[2 * i + 0] = x.x; r.w[2 * i + 1] = x.y;
    }
  } else {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(p);
#pragma unroll
    for (int i = 0; i < NDW; ++i) r.w[i] = src[i];
  }
  return r;
}

// Same as load_hvec, with the non-temporal hint: K/V are streamed once per
// call, so they should not displace the reused lines (q, block_table,
// partials) in the caches.
template <int NDW>
__device__ __forceinline__ HVec<NDW> load_hvec_stream(const _Float16* p) {
  HVec<NDW> r;
  if constexpr (NDW % 4 == 0) {
#pragma unroll
    for (int i = 0; i < NDW / 4; ++i) {
      const u4_t x = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(p) + i);
      r.w[4 * i + 0] = x[0]; r.w[4 * i + 1] = x[1]; r.w[4 * i + 2] = x[2]; r.w[4 * i + 3] = x[3];
    }
  } else if constexpr (NDW % 2 == 0) {
#pragma unroll
    for (int i = 0; i < NDW / 2; ++i) {
      const u2_t x = __builtin_nontemporal_load(reinterpret_cast<const u2_t*>(p) + i);
      r.w[2 * i + 0] = x[0]; r.w[2 * i + 1] = x[1];
    }
  } else if constexpr (NDW % 3 == 0) {
    // head_dim 96: 12-byte row segments, one 3-dword load each.
#pragma unroll
    for (int i = 0; i < NDW / 3; ++i) {
      const u3_t x = __builtin_nontemporal_load(reinterpret_cast<const u3_t*>(p) + i);
      r.w[3 * i + 0] = x[0]; r.w[3 * i + 1] = x[1]; r.w[3 * i + 2] = x[2];
    }
  } else {
#pragma unroll
    for (int i = 0; i < NDW; ++i) r.w[i] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p) + i);
  }
  return r;
}

// Raw buffer resource over [base, base + bytes) (gfx9 raw-buffer word 3:
// 32-bit data format, no swizzle); out-of-range accesses are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// Device-scope (SC1) accesses: coherent across all CUs and XCDs without
// cache maintenance instructions.
constexpr int kCachePolicyDevice = 16;  // SC1
typedef int32_t i2_t __attribute__((ext_vector_type(2)));
typedef int32_t i4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void store_device(__amdgpu_buffer_rsrc_t r, uint32_t off, f4_t v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i4_t, v), r, off, 0, kCachePolicyDevice);
}
__device__ __forceinline__ void store_device(__amdgpu_buffer_rsrc_t r, uint32_t off, float2 v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i2_t, v), r, off, 0, kCachePolicyDevice);
}
__device__ __forceinline__ f4_t load_device_f4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kCachePolicyDevice));
}
__device__ __forceinline__ float2 load_device_f2(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kCachePolicyDevice));
}

// Folds (m_s, l_s, O_s) into (m, l, acc), with its rounding spelled out: of a
// sum of two products the compiler may fuse either one, and not the same one
// wherever it compiles the fold, but a unit folded by all its workgroups and
// one folded by its last arrival have to give the same bits.
__device__ __forceinline__ void fold_state(float ms, float ls, f4_t os, float& m, float& l, f4_t& acc) {
  const float m_new = fmaxf(m, ms);
  const float alpha = exp2_fast(m - m_new);  // 0 while m is -inf
  const float beta = exp2_fast(ms - m_new);
  l = __builtin_fmaf(l, alpha, ls * beta);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(acc[i], alpha, os[i] * beta);
  m = m_new;
}

// N consecutive splits' partials of one (row, 4 columns) element, loaded
// with device-scope loads (the (m, l) pairs first, in split order, then the
// O vectors) and folded in split order:
//   m' = max(m, m_s),  l' = l 2^(m - m') + l_s 2^(m_s - m'),
//   acc' = acc 2^(m - m') + O_s 2^(m_s - m').
// Every load is unconditional: offsets past the unit's region read as zeros
// (buffer range check) and are not folded, so the loads of a batch need no
// branch and each fold step waits only for its own split's data.
template <int N>
struct MergeBatch {
  float2 ml[N];
  f4_t o[N];
  // Entry sp0 + j sits in split slot (sp0 + j) * stride.
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t o_rsrc, __amdgpu_buffer_rsrc_t ml_rsrc, int sp0,
                                       int stride, int gqa, int row, int col, int d) {
#pragma unroll
    for (int j = 0; j < N; ++j) ml[j] = load_device_f2(ml_rsrc, (uint32_t)((sp0 + j) * stride * gqa + row) * 8u);
#pragma unroll
    for (int j = 0; j < N; ++j)
      o[j] = load_device_f4(o_rsrc, ((uint32_t)((sp0 + j) * stride * gqa + row) * (uint32_t)d + col) * 4u);
  }
  // Entries at or past `end`, inside the unit's region, load as zeros.
  __device__ __forceinline__ void load_below(__amdgpu_buffer_rsrc_t o_rsrc, __amdgpu_buffer_rsrc_t ml_rsrc, int sp0,
                                             int end, int gqa, int row, int col, int d) {
    constexpr uint32_t kPast = 0x7ffffff0u;  // past any region
#pragma unroll
    for (int j = 0; j < N; ++j)
      ml[j] = load_device_f2(ml_rsrc, sp0 + j < end ? (uint32_t)((sp0 + j) * gqa + row) * 8u : kPast);
#pragma unroll
    for (int j = 0; j < N; ++j)
      o[j] = load_device_f4(o_rsrc, sp0 + j < end ? ((uint32_t)((sp0 + j) * gqa + row) * (uint32_t)d + col) * 4u : kPast);
  }
  // Entries at or past `end` fold with m_s = -inf, i.e. weight 0 (their
  // loads read zeros: they lie past the unit's region): the fold has no
  // branch, so the compiler cannot sink a load into a conditional step and
  // serialise the round trips.  The first entry always exists, so m is
  // finite before any such step and alpha stays 1.
  __device__ __forceinline__ void fold(int sp0, int end, float& m, float& l, f4_t& acc) const {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      // Every published split is non-empty, so its m is finite.
      const float ms = sp0 + j < end ? ml[j].x : kNegInf;
      const float m_new = fmaxf(m, ms);
      const float alpha = exp2_fast(m - m_new);  // 0 while m is -inf
      const float beta = exp2_fast(ms - m_new);
      l = l * alpha + ml[j].y * beta;
      acc = acc * alpha + o[j] * beta;
      m = m_new;
    }
  }
  // The same, one fold_state() after the other.
  __device__ __forceinline__ void fold_states(int sp0, int end, float& m, float& l, f4_t& acc) const {
#pragma unroll
    for (int j = 0; j < N; ++j) fold_state(sp0 + j < end ? ml[j].x : kNegInf, ml[j].y, o[j], m, l, acc);
  }
};

// Folds entries [first, first + count) of one element (entry i in split
// slot i * stride), one memory round trip per batch: 4, 8 or 16 entries for
// counts up to 4, 8 and 16, batches of 16 beyond.  Entries a batch reads
// past the count must lie past the unit's region (they read zeros).
__device__ __forceinline__ void merge_partials(__amdgpu_buffer_rsrc_t o_rsrc, __amdgpu_buffer_rsrc_t ml_rsrc,
                                               int first, int count, int stride, int gqa, int row, int col, int d,
                                               float& m, float& l, f4_t& acc) {
  const int end = first + count;
  if (count <= 4) {
    MergeBatch<4> p;
    p.load(o_rsrc, ml_rsrc, first, stride, gqa, row, col, d);
    p.fold(first, end, m, l, acc);
    return;
  }
  if (count <= 8) {
    MergeBatch<8> p;
    p.load(o_rsrc, ml_rsrc, first, stride, gqa, row, col, d);
    p.fold(first, end, m, l, acc);
    return;
  }
  for (int sp0 = first; sp0 < end; sp0 += 16) {
    MergeBatch<16> p;
    p.load(o_rsrc, ml_rsrc, sp0, stride, gqa, row, col, d);
    p.fold(sp0, end, m, l, acc);
  }
}

// Folds entries [first, end) of one element in batches of 4, to a state of
// its own.
__device__ __forceinline__ void fold_run(__amdgpu_buffer_rsrc_t o_rsrc, __amdgpu_buffer_rsrc_t ml_rsrc, int first,
                                         int end, int gqa, int row, int col, int d, float& m, float& l, f4_t& acc) {
  m = kNegInf;
  l = 0.f;
  acc = (f4_t)0.f;
  for (int sp0 = first; sp0 < end; sp0 += 4) {
    MergeBatch<4> p;
    p.load_below(o_rsrc, ml_rsrc, sp0, end, gqa, row, col, d);
    p.fold_states(sp0, end, m, l, acc);
  }
}

// Reads an int32 at a wave-uniform address with a scalar load (constant
// address space): the value lands in an SGPR and its wait counts on the
// LDS/scalar counter, so it never has to drain the K/V vector loads in
// flight, as a vector load of the same word would (vector loads complete in
// order).  The memory must stay unchanged while the kernel runs.
__device__ __forceinline__ int32_t load_uniform_i32(const int32_t* p) {
  return *(const __attribute__((address_space(4))) int32_t*)p;
}

__device__ __forceinline__ int clamp_page(int phys, int64_t num_pages) {
  // Keeps every access inside the cache for an invalid block_table entry
  // (the reference documents valid ids as a precondition and does not
  // check them on the device; here a bad id reads page 0 instead of
  // faulting).
  return (phys < 0 || (int64_t)phys >= num_pages) ? 0 : phys;
}

// ---------------------------------------------------------------------------
// Per-wave state handed to the workgroup merge, written to LDS in one format
// for both engines:  sm_ml[w*16 + row] = (m, l),
// sm_o[(w*gqa + row)*wave_row_floats<D>() + d].  The 16-byte row pad puts
// the 16 rows a wave writes with one instruction in different LDS banks.
// ---------------------------------------------------------------------------
template <int D>
constexpr int wave_row_floats() { return D + 4; }

// Bytes per token row of a wave's K staging tile in LDS (16 rows): the row
// plus 16 bytes of padding, so the 16-row column reads of the MFMA operand
// fall in different banks.
template <int D>
constexpr int k_stage_row_bytes() { return D * 2 + 16; }
template <int D>
constexpr int k_stage_bytes() { return 16 * k_stage_row_bytes<D>(); }

// With whole-page blocks, the page id of the wave's first block is read
// before the sequence length is known, so its latency overlaps the
// seq_lens read (the column is clamped into the table; its value is only
// used when the block exists).
__device__ __forceinline__ int first_page_id(const Phase1Args& a, const int32_t* ids_row, int64_t ids_stride,
                                             int col_max, int p_first, int wave) {
  if (col_max < 0) return 0;
  const int col = min(p_first + block_page(a, wave), col_max);
  return load_uniform_i32(ids_row + (int64_t)col * ids_stride);
}

// Block-addressing modes of the MFMA wave loop (template parameter MODE):
//   kModeGeneric  any other page size (>= 3): a block spans up to 6 pages;
//   kModeUniform  page_size % 16 == 0: a 16-token block lies in one page;
//   kModeSubpage + s  page_size = 2^s < 16: a block covers 16 >> s whole
//                 pages (items start on page boundaries).
constexpr int kModeGeneric = 0;
constexpr int kModeUniform = 1;
constexpr int kModeSubpage = 2;

// Element formats (template parameter KVF of the MFMA engine): fp16; an
// OCP fp8 cache format, widened to fp16 in registers where compute() uses a
// block, so that everything downstream (K staging, both MFMAs, the softmax)
// is the fp16 path; or bfloat16 q, caches and output, which run the same
// path on bf16 MFMAs (P rounded to bf16, as fp16 P is to fp16).
constexpr int kKvF16 = 0;
constexpr int kKvE4M3 = 1;   // float8_e4m3fn caches, fp16 q and output
constexpr int kKvE5M2 = 2;   // float8_e5m2 caches, fp16 q and output
constexpr int kKvBF16 = 3;   // bfloat16 q, caches and output
constexpr int kKvE4M3B = 4;  // float8_e4m3fn caches, bfloat16 q and output
constexpr int kKvE5M2B = 5;  // float8_e5m2 caches, bfloat16 q and output

template <int KVF>
constexpr bool kv_is_fp8() { return KVF == kKvE4M3 || KVF == kKvE5M2 || KVF == kKvE4M3B || KVF == kKvE5M2B; }
template <int KVF>
constexpr bool kv_is_e4m3() { return KVF == kKvE4M3 || KVF == kKvE4M3B; }
// bfloat16 q, P and output (and MFMAs); fp16 otherwise.
template <int KVF>
constexpr bool q_is_bf16() { return KVF == kKvBF16 || KVF == kKvE4M3B || KVF == kKvE5M2B; }
template <int KVF>
constexpr int kv_elem_bytes() { return kv_is_fp8<KVF>() ? 1 : 2; }

// One 16x16x16 MFMA step on 16-bit operands held as fp16 vectors: fp16, or
// the bit patterns of bfloat16 values (q_is_bf16).
template <int KVF>
__device__ __forceinline__ f4_t mfma16(h4_t a, h4_t b, f4_t c) {
  if constexpr (q_is_bf16<KVF>()) {
    typedef short s4_t __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4_t, a), __builtin_bit_cast(s4_t, b), c,
                                                     0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  }
}

// x rounded (to nearest even) to the output format, as 16 bits in an fp16
// slot: fp16, or bfloat16 (q_is_bf16).
template <int KVF>
__device__ __forceinline__ _Float16 round16(float x) {
  if constexpr (q_is_bf16<KVF>())
    return __builtin_bit_cast(_Float16, (__bf16)x);
  else
    return (_Float16)x;
}

// Four fp8 codes (one dword, element i in byte i) as four 16-bit values
// (two dwords: elements 0-1 in lo, 2-3 in hi) in the compute format, fp16
// or bfloat16, with gfx950's scaled conversions (v_cvt_scalef32_pk_f16_fp8 /
// _bf8, or _pk_bf16_fp8 / _bf8, one per pair).  Their scale operand acts
// through its exponent only, so it is 1 here and the launch folds the
// caller's k_scale / v_scale into the softmax scale and the output
// normalisation.  At scale 1 every code converts exactly, NaN codes to NaNs
// (every e4m3fn value and every e5m2 value is an fp16 and a bf16 value).
template <int KVF>
__device__ __forceinline__ void fp8x4_to_16x4(uint32_t w, uint32_t& lo, uint32_t& hi) {
  if constexpr (q_is_bf16<KVF>()) {
    typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
    b2_t a, b;
    if constexpr (kv_is_e4m3<KVF>()) {
      a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false);
      b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true);
    } else {
      a = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.0f, false);
      b = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.0f, true);
    }
    lo = __builtin_bit_cast(uint32_t, a);
    hi = __builtin_bit_cast(uint32_t, b);
  } else {
    h2_t a, b;
    if constexpr (kv_is_e4m3<KVF>()) {
      a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false);
      b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true);
    } else {
      a = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w, 1.0f, false);
      b = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w, 1.0f, true);
    }
    lo = __builtin_bit_cast(uint32_t, a);
    hi = __builtin_bit_cast(uint32_t, b);
  }
}

// head_dim 256 keeps the Q^T operand in LDS instead of 32 VGPRs per lane
// (with it in registers the kernel spilled 25-38 VGPRs to scratch inside
// the streaming loop).  One padded 16-row copy per workgroup: every lane
// writes its own fragments and reads back only those addresses, so no
// barrier is needed (the waves write identical values).
template <int D>
constexpr bool q_in_lds() { return D >= 256; }

// Wave-wide integer reductions: DPP within each 16-lane row, then the four
// row results combined through readlane (wave-uniform result).
__device__ __forceinline__ int row16_sum_i32(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
  x += __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
  x += __builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, false);  // row_half_mirror
  x += __builtin_amdgcn_update_dpp(0, x, 0x140, 0xF, 0xF, false);  // row_mirror
  return x;
}

__device__ __forceinline__ int wave_sum_i32(int x) {
  x = row16_sum_i32(x);
  return __builtin_amdgcn_readlane(x, 0) + __builtin_amdgcn_readlane(x, 16) + __builtin_amdgcn_readlane(x, 32) +
         __builtin_amdgcn_readlane(x, 48);
}

__device__ __forceinline__ int wave_max_i32(int x) {
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x140, 0xF, 0xF, false));
  return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
             max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

// Inclusive prefix sum over the 64 lanes: row_shr steps (bound_ctrl shifts
// in zeros) scan each 16-lane row, then each row adds the totals of the rows
// before it.
__device__ __forceinline__ int wave_incl_scan_i32(int x, int lane) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);  // row_shr:8
  const int r0 = __builtin_amdgcn_readlane(x, 15);
  const int r1 = __builtin_amdgcn_readlane(x, 31);
  const int r2 = __builtin_amdgcn_readlane(x, 47);
  const int row = lane >> 4;
  return x + (row >= 1 ? r0 : 0) + (row >= 2 ? r1 : 0) + (row >= 3 ? r2 : 0);
}

// CSR row of sequence b: first page-id offset, page count and tokens.  The
// offsets are clamped into indices[0, max_pages) (max_pages holds the
// length of `indices` in CSR mode), so a malformed indptr cannot make the
// kernel read outside the array; last_page_len is clamped to the page.
__device__ __forceinline__ void csr_row(const Phase1Args& a, int b, int* row, int* pages, int* len) {
  const int r0 = min(max(a.indptr[b], 0), a.max_pages);
  const int r1 = min(max(a.indptr[b + 1], r0), a.max_pages);
  *row = r0;
  *pages = r1 - r0;
  *len = *pages > 0 ? (*pages - 1) * a.ps + min(max(a.lpl[b], 1), a.ps) : 0;
}

// Sequence table spread over the wave: lane l holds sequences l + 64k,
// k < NK (NK = 1 for batches up to 64, else 4).
template <int NK>
struct SeqTable {
  int len[NK];    // tokens (0 past the batch)
  int pages[NK];  // pages in use
  int row[NK];    // CSR: offset of the sequence's page ids in `indices`
};

// Raw words of the sequence table for up to 256 sequences (lane l holds
// sequences l + 64k): CSR indptr[b], indptr[b + 1] and last_page_len[b];
// the dense table reads seq_lens[b] into all three.  A workgroup issues
// these loads before its first page-id read and uses them after it, so the
// two share one memory round trip; every load is unconditional (a lane past
// the batch re-reads the last sequence's words), so no branch has to wait
// for any of them.
struct SeqRaw {
  int r0[4], r1[4], r2[4];
};

__device__ __forceinline__ SeqRaw issue_seq_table(const Phase1Args& a, int lane) {
  SeqRaw r;
  const int32_t* p0 = a.csr ? a.indptr : a.sl;
  const int32_t* p1 = a.csr ? a.indptr + 1 : a.sl;
  const int32_t* p2 = a.csr ? a.lpl : a.sl;
  const int64_t stride = a.csr ? 1 : a.ssl;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t off = (int64_t)min(lane + 64 * k, a.batch - 1) * stride;
    r.r0[k] = p0[off];
    r.r1[k] = p1[off];
    r.r2[k] = p2[off];
  }
  return r;
}

template <int NK>
__device__ __forceinline__ SeqTable<NK> seq_table(const Phase1Args& a, const SeqRaw& r, int lane) {
  SeqTable<NK> t;
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const bool in = lane + 64 * k < a.batch;
    int len, pages, row = 0;
    if (a.csr) {
      row = min(max(r.r0[k], 0), a.max_pages);
      pages = min(max(r.r1[k], row), a.max_pages) - row;
      len = pages > 0 ? (pages - 1) * a.ps + min(max(r.r2[k], 1), a.ps) : 0;
    } else {
      len = max(r.r0[k], 0);
      pages = min(pages_for(a, len), a.max_pages);
    }
    t.len[k] = in ? len : 0;
    t.pages[k] = in ? pages : 0;
    t.row[k] = in ? row : 0;
  }
  return t;
}

}  // namespace pad

#endif  // PA_DEVICE_H_
