// pa_range.hip - gfx950 paged-attention decode over equal page ranges.
//
// The kernel for bandwidth-bound calls whose kv heads come in groups (or one
// by one) and whose split count is left to the launcher.  Two things bound
// such calls in the per-(sequence, kv head) kernel of pa_decode.hip, and
// this one is built around both:
//
//  * DRAM locality.  A kv head's slice of a token row is 128 or 256 bytes of
//    a row of hkv such slices.  Workgroups that stream one head each read the
//    slices of a row at different times, from the few channels that head's
//    addresses fall into.  Here a workgroup's waves take the (up to 4) kv
//    heads of a head group side by side, each wave one head over the same
//    tokens, so neighbouring slices are read together.  A read-only probe of
//    the access pattern (8 kv heads, pages of 16 tokens): 1 x 131072 tokens
//    6.3 -> 6.85 TB/s with 256-byte slices and 5.7 -> 6.4-6.6 with 128-byte
//    ones; 64 x 8192 tokens 6.5 -> 6.9 and 6.2 -> 6.9 TB/s.
//  * Balance.  The pages of all (sequence, head group) units are laid end to
//    end and cut into one equal range per workgroup, instead of cutting each
//    unit into chunks: no chunk is rounded up, so every CU ends at the same
//    time.  Each unit counts some pages more than it has, at its front: the
//    time a workgroup takes from one unit to the next.  A workgroup walks its
//    range unit by unit ("segments"); a unit that lies inside one range is
//    written straight to the output, one that spans several has one partial
//    per range, folded by the last workgroup of the unit to arrive
//    (pa_decode.hip's protocol).
//
// See range_wave_loop for the streaming loop.

#include "pa_range.h"

namespace pad {

// NDW dwords of a token row in NSEG equal segments 16 lanes apart
// (RowLayout), loaded with the non-temporal hint: from a wave-uniform base
// with a 32-bit lane offset, or from a lane's own address.
constexpr int kCachePolicyStream = 2;  // NT
template <int NDW, int NSEG>
__device__ __forceinline__ HVec<NDW> load_row_buffer(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  constexpr int W = NDW / NSEG;
  HVec<NDW> x;
#pragma unroll
  for (int sg = 0; sg < NSEG; ++sg) {
    const uint32_t o = off + sg * 64 * W;
    if constexpr (W == 4) {
      const u4_t v = __builtin_bit_cast(u4_t, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, kCachePolicyStream));
#pragma unroll
      for (int w = 0; w < W; ++w) x.w[sg * W + w] = v[w];
    } else if constexpr (W == 3) {
      const u3_t v = __builtin_bit_cast(u3_t, __builtin_amdgcn_raw_buffer_load_b96(r, o, 0, kCachePolicyStream));
#pragma unroll
      for (int w = 0; w < W; ++w) x.w[sg * W + w] = v[w];
    } else if constexpr (W == 2) {
      const u2_t v = __builtin_bit_cast(u2_t, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, kCachePolicyStream));
#pragma unroll
      for (int w = 0; w < W; ++w) x.w[sg * W + w] = v[w];
    } else {
      static_assert(W == 1, "segment width");
      x.w[sg] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, o, 0, kCachePolicyStream);
    }
  }
  return x;
}
template <int NDW, int NSEG>
__device__ __forceinline__ HVec<NDW> load_row(const char* p) {
  constexpr int W = NDW / NSEG;
  HVec<NDW> x;
#pragma unroll
  for (int sg = 0; sg < NSEG; ++sg) {
    const HVec<W> v = load_hvec_stream<W>(reinterpret_cast<const _Float16*>(p + sg * 64 * W));
#pragma unroll
    for (int w = 0; w < W; ++w) x.w[sg * W + w] = v.w[w];
  }
  return x;
}

// The same row into LDS, each segment as one store where its size allows.
template <int NDW, int NSEG>
__device__ __forceinline__ void stage_row(char* dst, const HVec<NDW>& x) {
  constexpr int W = NDW / NSEG;
#pragma unroll
  for (int sg = 0; sg < NSEG; ++sg) {
    char* p = dst + sg * 64 * W;
    if constexpr (W == 4) {
      *reinterpret_cast<u4_t*>(p) = u4_t{x.w[sg * W], x.w[sg * W + 1], x.w[sg * W + 2], x.w[sg * W + 3]};
    } else if constexpr (W == 2) {
      *reinterpret_cast<u2_t*>(p) = u2_t{x.w[sg * W], x.w[sg * W + 1]};
    } else {
#pragma unroll
      for (int w = 0; w < W; ++w) reinterpret_cast<uint32_t*>(p)[w] = x.w[sg * W + w];
    }
  }
}

// How a token row of a cache is read: lane r16 of a 16-lane group takes NSEG
// segments of SEGB bytes (SE elements), so that the group reads 16 * SEGB
// contiguous bytes per load instruction.  Element dt of the lane is head_dim
// slot (dt / SE) * 16 * SE + r16 * SE + dt % SE.  One segment up to 256-byte
// rows; 512-byte rows (head_dim 256, 16-bit) are two 256-byte halves.
template <int D, int KVF>
struct RowLayout {
  static constexpr int ES = kv_elem_bytes<KVF>();
  static constexpr int LANE_BYTES = D * ES / 16;
  static constexpr int SEGB = LANE_BYTES > 16 ? 16 : LANE_BYTES;
  static constexpr int NSEG = LANE_BYTES / SEGB;
  static constexpr int SE = SEGB / ES;
  static constexpr int NDW = LANE_BYTES / 4;  // dwords per lane per row, as stored
  static constexpr int KROW = D * ES + 16;    // bytes per row of the wave's K stage (padded)
};

// 16-token blocks that a wave computes together (see wave_loop_mfma): two, up
// to head_dim 128.  Two tiles of two blocks of 512-byte rows would not fit the
// register file (fp8 caches go along).  Ranges and waves follow the bytes of
// the caches, so fp8 results equal 16-bit ones on the same values to rounding.
template <int D>
constexpr int tile_blocks() { return D <= 128 ? 2 : 1; }

// N 16-token blocks of K and V in registers as loaded: lane (g, r16) holds
// its segments of token rows 4g+i of each block (fp8 caches: codes, widened
// only where compute() uses them).
template <int N, int NDW>
struct KVTile {
  HVec<NDW> k[N][4];
  HVec<NDW> v[N][4];
};

// Page ids of N blocks and the slot of each block's first token in its first
// page.  NID ids per block: one, or those of a lane's own token rows (page
// sizes that do not hold whole 16-token blocks).
template <int N, int NID>
struct TileIds {
  int id[N][NID];
  int slot[N];
};

// The 16x16x32 form does the work of two 16x16x16 steps (8 operand elements
// per lane).
template <int KVF>
__device__ __forceinline__ f4_t mfma32(h8_t a, h8_t b, f4_t c) {
  if constexpr (q_is_bf16<KVF>()) {
    typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8_t, a), __builtin_bit_cast(b8_t, b), c, 0, 0,
                                                   0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
}

// Two 16-bit values in a dword (a in the low half), and two floats rounded
// to the compute format in one.
__device__ __forceinline__ uint32_t pack_pair(_Float16 a, _Float16 b) {
  return __builtin_bit_cast(uint32_t, h2_t{a, b});
}
template <int KVF>
__device__ __forceinline__ uint32_t pack16(float a, float b) {
  return pack_pair(round16<KVF>(a), round16<KVF>(b));
}

// One wave's part of a segment: the 16-token blocks wave, wave + nw, ... of
// tokens [t_begin, t_end) for kv head kvh.  Tiles of one or two blocks
// (tile_blocks) are double buffered in registers: the next tile's loads are
// issued before the current one is computed, and stay in flight across it
// (every wait in the steady-state loop leaves them outstanding).  Scores are
// S^T = K.Q^T and the output O^T = V^T.P^T on 16x16x32 MFMAs; with two blocks
// the PV product contracts 32 tokens (4 of each block per lane group), half
// the matrix instructions of two 16-token steps.
template <int D, int MODE, int KVF = kKvF16>
__device__ __forceinline__ void range_wave_loop(const Phase1Args& a, int phys_first, const int32_t* bt_row,
                                                int64_t ids_stride, int b, int kvh, int t_begin, int t_end,
                                                int nblk, int wave, int nw, int slot, int lane, float2* sm_ml,
                                                float* sm_o, char* k_stage, char* q_stage) {
  using R = RowLayout<D, KVF>;
  constexpr int DK = D / 32;      // 32-wide head_dim steps of K.Q^T
  constexpr int DT = D / 16;      // PV output tiles; V elements per lane per token
  constexpr int NB = tile_blocks<D>();
  constexpr int ES = R::ES;
  constexpr int NDW = R::NDW;
  constexpr int SE = R::SE;
  constexpr bool FP8 = kv_is_fp8<KVF>();
  static_assert(!FP8 || D % 64 == 0, "fp8 caches: head_dim a multiple of 64");
  const int g = lane >> 4;
  const int r16 = lane & 15;
  const bool row_ok = r16 < a.gqa;
  // The wave's Q^T operand (B of S^T = K.Q^T: row r16, head_dim slots
  // kp*32 + g*8 + [0,8)), loaded after the first K/V block is in flight.
  h8_t qv[q_in_lds<D>() ? 1 : DK];
  auto q_slot = [&](int kp) -> h8_t* {
    return reinterpret_cast<h8_t*>(q_stage + r16 * k_stage_row_bytes<D>() + (kp * 32 + g * 8) * 2);
  };
  auto load_q = [&]() {
    const _Float16* qrow = a.q + (int64_t)b * a.sqb + (int64_t)(kvh * a.gqa + (row_ok ? r16 : 0)) * a.sqh;
#pragma unroll
    for (int kp = 0; kp < DK; ++kp) {
      const h8_t x = *reinterpret_cast<const h8_t*>(qrow + kp * 32 + g * 8);
      if constexpr (q_in_lds<D>())
        *q_slot(kp) = row_ok ? x : (h8_t)0;
      else
        qv[kp] = row_ok ? x : (h8_t)0;
    }
  };

  float m_run = kNegInf;
  f4_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = (f4_t)0.f;
  // Row sums of P come from one more MFMA with an operand of ones (row 0 of
  // the result; the four rows are alike).
  f4_t o_l = (f4_t)0.f;
  const _Float16 one16 = round16<KVF>(1.0f);

  const char* k_head = reinterpret_cast<const char*>(a.k) + (int64_t)kvh * a.skh * ES;
  const char* v_head = reinterpret_cast<const char*>(a.v) + (int64_t)kvh * a.svh * ES;
  const uint32_t page_limit = (uint32_t)min(a.num_pages, (int64_t)0x7fffffff);
  auto clamp_id = [&](int id) -> uint32_t { return (uint32_t)id < page_limit ? (uint32_t)id : 0u; };
  // Lane byte offsets inside a 16-token slab of one page (loop invariant).
  // K and V are both read as whole token rows: lane (g, r16) reads row 4g+i
  // (RowLayout), so one load instruction covers four rows.  K then goes
  // through LDS into the MFMA operand layout (token per lane%16).
  // Sub-page blocks: token 4g+i sits in slot (4g+i) mod page_size of its
  // page (blocks start on page boundaries), again loop invariant.
  constexpr int SUB_SHIFT = MODE >= kModeSubpage ? MODE - kModeSubpage : 0;
  uint32_t koff[4], voff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = MODE == kModeUniform ? 4 * g + i : (MODE >= kModeSubpage ? (4 * g + i) & ((1 << SUB_SHIFT) - 1) : 0);
    koff[i] = (uint32_t)((int64_t)row * a.sks * ES + r16 * R::SEGB);
    voff[i] = (uint32_t)((int64_t)row * a.svs * ES + r16 * R::SEGB);
  }

  // Position of the wave's next block: page (from the item's first) and slot
  // of its first token.  Blocks of a wave are nw apart.
  // (Quotients come out of vector registers: as scalars they keep the page
  // ids and bases that follow from them scalar.)
  auto scalar = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  const int p_first = scalar(page_of(a, t_begin));
  const int p_last = scalar(t_end > t_begin ? page_of(a, t_end - 1) : p_first);
  int cur_page = scalar(page_of(a, wave * kBlockTokens));
  int cur_slot = wave * kBlockTokens - cur_page * a.ps;
  const int step_pages = scalar(page_of(a, nw * kBlockTokens));
  const int step_slots = nw * kBlockTokens - step_pages * a.ps;
  auto advance = [&]() {
    cur_page += step_pages;
    cur_slot += step_slots;
    if (cur_slot >= a.ps) {
      cur_slot -= a.ps;
      ++cur_page;
    }
  };

  // Page ids run one tile ahead of the K/V loads that use them.
  //  * Whole-page blocks: one id per block, a scalar load (it waits on the
  //    scalar counter, so it never drains the K/V loads in flight).
  //  * Other page sizes: each lane loads the ids of its own four token rows
  //    (1, 2 or 4 of them per block).  They are issued before the K/V loads
  //    of the tile ahead of theirs: vector loads return in order, so using
  //    them leaves those K/V loads in flight.  An arbitrary page size finds
  //    each row's page and slot by an exact float-reciprocal division of its
  //    offset from the block's first page ((pos + 0.5) / ps is never within
  //    0.5 / ps of an integer).
  // Columns past the item's last page are clamped to it (its tokens are
  // masked).
  constexpr int NID = MODE == kModeUniform ? 1 : (MODE == kModeGeneric || SUB_SHIFT == 0 ? 4 : (SUB_SHIFT == 1 ? 2 : 1));
  using Ids = TileIds<NB, NID>;
  const float inv_ps = 1.0f / (float)a.ps;
  auto page_in_block = [&](int pos) { return (int)(((float)pos + 0.5f) * inv_ps); };
  // Fetches the ids of the wave's next block as entry s of x, and moves past it.
  auto fetch_block = [&](Ids& x, int s) {
    const int p0 = p_first + cur_page;
    x.slot[s] = cur_slot;
    if constexpr (MODE == kModeUniform) {
      x.id[s][0] = load_uniform_i32(bt_row + (int64_t)min(p0, p_last) * ids_stride);
    } else {
#pragma unroll
      for (int k = 0; k < NID; ++k) {
        int col = p0;
        if constexpr (MODE >= kModeSubpage)
          col += (4 * g + k * (4 / NID)) >> SUB_SHIFT;
        else
          col += page_in_block(cur_slot + 4 * g + k);
        x.id[s][k] = bt_row[(int64_t)min(col, p_last) * ids_stride];
      }
    }
    advance();
  };
  auto fetch_ids = [&](Ids& x) {
#pragma unroll
    for (int s = 0; s < NB; ++s) fetch_block(x, s);
  };

  // Issues the K/V loads of one block.
  auto load_rows = [&](HVec<NDW> (&tk)[4], HVec<NDW> (&tv)[4], const int (&id)[NID], int slot) {
    if constexpr (MODE == kModeUniform) {
      // page_size % 16 == 0: the block lies in one page, so its base is
      // wave-uniform: buffer loads with a scalar base and 32-bit lane offsets.
      const uint64_t phys = clamp_id(id[0]);
      const char* kb = k_head + (phys * (uint64_t)a.skp + (uint64_t)((int64_t)slot * a.sks)) * ES;
      const char* vb = v_head + (phys * (uint64_t)a.svp + (uint64_t)((int64_t)slot * a.svs)) * ES;
      const __amdgpu_buffer_rsrc_t kr = make_rsrc(kb, 0xffffffffu), vr = make_rsrc(vb, 0xffffffffu);
#pragma unroll
      for (int i = 0; i < 4; ++i) tk[i] = load_row_buffer<NDW, R::NSEG>(kr, koff[i]);
#pragma unroll
      for (int i = 0; i < 4; ++i) tv[i] = load_row_buffer<NDW, R::NSEG>(vr, voff[i]);
    } else {
      const uint64_t kpage = (uint64_t)(a.skp * ES), vpage = (uint64_t)(a.svp * ES);
      auto row_addr = [&](const char* head, uint64_t page_bytes, int64_t slot_bytes, uint32_t off, int i) {
        const char* p = head + (uint64_t)clamp_id(id[i * NID / 4]) * page_bytes + off;
        if constexpr (MODE == kModeGeneric) {
          const int pos = slot + 4 * g + i;
          p += (int64_t)(pos - page_in_block(pos) * a.ps) * slot_bytes;
        }
        return p;
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) tk[i] = load_row<NDW, R::NSEG>(row_addr(k_head, kpage, a.sks * ES, koff[i], i));
#pragma unroll
      for (int i = 0; i < 4; ++i) tv[i] = load_row<NDW, R::NSEG>(row_addr(v_head, vpage, a.svs * ES, voff[i], i));
    }
  };

  // One tile: N blocks, first block jb, the second nw later.  masked: the
  // tile may hold the item's last block, whose tail is masked.
  auto compute = [&](auto& t, auto masked_c, int jb) {
    constexpr int N = sizeof(t.k) / sizeof(t.k[0]);
    constexpr bool MASKED = decltype(masked_c)::value;
    // K rows -> LDS (row 4g+i, the lane's segments), then the MFMA A operand back
    // out: lane (g, r16) takes token r16, head_dim kp*32 + g*8 + [0, 8).
    // LDS accesses of one wave complete in order, so the reads see the
    // writes, and the next block's writes follow these reads.
    float x[N][4];
    f4_t sacc[N];
#pragma unroll
    for (int s = 0; s < N; ++s) {
#pragma unroll
      for (int i = 0; i < 4; ++i) stage_row<NDW, R::NSEG>(k_stage + (4 * g + i) * R::KROW + r16 * R::SEGB, t.k[s][i]);
      const char* src = k_stage + r16 * R::KROW + g * 8 * ES;
      sacc[s] = (f4_t)0.f;
#pragma unroll
      for (int kp = 0; kp < DK; ++kp) {
        h8_t kk;
        if constexpr (FP8) {
          const uint2 c = *reinterpret_cast<const uint2*>(src + kp * 32);
          u4_t w;
          uint32_t lo, hi;
          fp8x4_to_16x4<KVF>(c.x, lo, hi);
          w[0] = lo; w[1] = hi;
          fp8x4_to_16x4<KVF>(c.y, lo, hi);
          w[2] = lo; w[3] = hi;
          kk = __builtin_bit_cast(h8_t, w);
        } else {
          kk = *reinterpret_cast<const h8_t*>(src + kp * 64);
        }
        h8_t qk;
        if constexpr (q_in_lds<D>())
          qk = *q_slot(kp);
        else
          qk = qv[kp];
        // S^T[token 4g+i][row r16] over head_dim.
        sacc[s] = mfma32<KVF>(kk, qk, sacc[s]);
      }
    }
#pragma unroll
    for (int s = 0; s < N; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) x[s][i] = sacc[s][i] * a.scale_log2;
    if constexpr (MASKED) {
#pragma unroll
      for (int s = 0; s < N; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool valid = t_begin + (jb + s * nw) * kBlockTokens + 4 * g + i < t_end;
          x[s][i] = valid ? x[s][i] : kNegInf;
#pragma unroll
          for (int w = 0; w < NDW; ++w)  // stale cache slots may hold NaN/Inf
            t.v[s][i].w[w] = valid ? t.v[s][i].w[w] : 0u;
        }
    }
    float bm = kNegInf;
#pragma unroll
    for (int s = 0; s < N; ++s) bm = fmaxf(bm, fmaxf(fmaxf(x[s][0], x[s][1]), fmaxf(x[s][2], x[s][3])));
    // Lazy rescaling: the reference m_run only moves when a score exceeds it
    // by more than kRescaleSlack (base-2 units), so weights stay <= 2^slack
    // and the O/l rescale is skipped (wave-uniformly) on most tiles.  Any
    // reference value gives the same O/l; partials carry it as their m.
    // Whether any score does needs no row maximum, only each lane's own; the
    // row's is formed when the reference moves.  Every tile holds at least
    // one valid token, so it is finite.
    if (__builtin_amdgcn_ballot_w64(bm > m_run + kRescaleSlack) != 0) {
      bm = fmaxf(bm, shfl_xor_f(bm, 16));
      bm = fmaxf(bm, shfl_xor_f(bm, 32));
      const float m_new = fmaxf(m_run, bm);
      const float alpha = exp2_fast(m_run - m_new);  // 0 on the first tile
      o_l[0] *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
      m_run = m_new;
    }
    // P^T in the B operand layout: the lane's 4N tokens (l accumulates the
    // same rounded weights P.V uses).
    uint32_t pw[2 * N];
#pragma unroll
    for (int s = 0; s < N; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        pw[2 * s + j] = pack16<KVF>(exp2_fast(x[s][2 * j] - m_run), exp2_fast(x[s][2 * j + 1] - m_run));
    // V^T as the A operand: for each PV tile dt, pairs of token rows.
    auto pv = [&](int s, int j, int dt) -> uint32_t {  // rows 2j, 2j+1 of block s
      if constexpr (FP8) {
        return 0u;
      } else {
        return __builtin_amdgcn_perm(t.v[s][2 * j + 1].w[dt / 2], t.v[s][2 * j].w[dt / 2],
                                     dt % 2 ? 0x07060302u : 0x05040100u);
      }
    };
    auto accumulate = [&](const uint32_t (&vw)[2 * N], f4_t& acc) {
      if constexpr (N == 2) {
        acc = mfma32<KVF>(__builtin_bit_cast(h8_t, u4_t{vw[0], vw[1], vw[2], vw[3]}),
                          __builtin_bit_cast(h8_t, u4_t{pw[0], pw[1], pw[2], pw[3]}), acc);
      } else {
        acc = mfma16<KVF>(__builtin_bit_cast(h4_t, u2_t{vw[0], vw[1]}), __builtin_bit_cast(h4_t, u2_t{pw[0], pw[1]}),
                          acc);
      }
    };
    {
      const uint32_t ones = pack_pair(one16, one16);
      uint32_t vw[2 * N];
#pragma unroll
      for (int j = 0; j < 2 * N; ++j) vw[j] = ones;
      accumulate(vw, o_l);
    }
    if constexpr (FP8) {
      // Codes of two rows interleaved bytewise before they are widened: one
      // byte permute gives two row pairs' codes, half the permutes of the
      // 16-bit form.
#pragma unroll
      for (int w = 0; w < NDW; ++w) {
        uint32_t vw[4][2 * N];  // [element 4w + e][row pair]
#pragma unroll
        for (int s = 0; s < N; ++s)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const uint32_t r0 = t.v[s][2 * j].w[w], r1 = t.v[s][2 * j + 1].w[w];
            fp8x4_to_16x4<KVF>(__builtin_amdgcn_perm(r1, r0, 0x05010400u), vw[0][2 * s + j], vw[1][2 * s + j]);
            fp8x4_to_16x4<KVF>(__builtin_amdgcn_perm(r1, r0, 0x07030602u), vw[2][2 * s + j], vw[3][2 * s + j]);
          }
#pragma unroll
        for (int e = 0; e < 4; ++e) accumulate(vw[e], o[4 * w + e]);
      }
    } else {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        uint32_t vw[2 * N];
#pragma unroll
        for (int s = 0; s < N; ++s)
#pragma unroll
          for (int j = 0; j < 2; ++j) vw[2 * s + j] = pv(s, j, dt);
        accumulate(vw, o[dt]);
      }
    }
  };

  // This wave's blocks are wave, wave+nw, ..., computed in tiles of NB; with
  // two per tile, an odd count starts with a tile of one.  The steady-state
  // loop issues the next tile's loads before computing the current one; only
  // the wave's last tile can hold the item's partial block.
  const int n_mine = scalar(wave < nblk ? (nblk - wave + nw - 1) / nw : 0);
  typedef KVTile<NB, NDW> Tile;
  struct No { enum { value = 0 }; };
  struct Yes { enum { value = 1 }; };
  Tile ta, tb;
  Ids ia, ib;
  // Loads one tile from `use`, whose ids have arrived, after issuing the
  // fetch of the next tile's ids.
  auto load = [&](Tile& t, const Ids& use, Ids& next) {
    if constexpr (MODE != kModeUniform) {
      fetch_ids(next);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < NB; ++s) load_rows(t.k[s], t.v[s], use.id[s], use.slot[s]);
    if constexpr (MODE == kModeUniform) fetch_ids(next);
    __builtin_amdgcn_sched_barrier(0);
  };
  if (n_mine > 0) {
    int jb = wave;
    const bool odd = NB == 2 && (n_mine & 1);
    const int tiles = n_mine / NB;
    // The first tile's loads are issued on one path, with the single block
    // before it where there is one: a join of two paths with loads in flight
    // would copy their registers, and so wait for them.
    KVTile<1, NDW> t1;
    if constexpr (MODE == kModeUniform) {
      ia.slot[0] = cur_slot;
      ia.id[0][0] = phys_first;
      advance();
      if (odd) {
        load_rows(t1.k[0], t1.v[0], ia.id[0], ia.slot[0]);
        fetch_block(ia, 0);
      }
      if constexpr (NB == 2) fetch_block(ia, 1);
    } else {
      Ids i1;
      if (odd) fetch_block(i1, 0);
      fetch_ids(ia);
      __builtin_amdgcn_sched_barrier(0);
      if (odd) load_rows(t1.k[0], t1.v[0], i1.id[0], i1.slot[0]);
    }
    if (tiles > 0) load(ta, ia, ib);
    load_q();
    if (odd) {
      compute(t1, Yes(), jb);
      jb += nw;
    }
    int it = 0;
    for (; it + 2 < tiles; it += 2) {
      load(tb, ib, ia);
      compute(ta, No(), jb);
      load(ta, ia, ib);
      compute(tb, No(), jb + NB * nw);
      jb += 2 * NB * nw;
    }
    if (it + 1 < tiles) {
      load(tb, ib, ia);
      compute(ta, No(), jb);
      compute(tb, Yes(), jb + NB * nw);
    } else if (it < tiles) {
      compute(ta, Yes(), jb);
    }
  }

  // The wave's state to LDS.  Lane (g, r16) owns O[row r16][dim(4g+i, dt)]: for
  // each i, NSEG runs of SE consecutive floats.
  auto o_slot = [&](int i, int dt) { return (dt / SE) * 16 * SE + (4 * g + i) * SE + dt % SE; };
  if (!row_ok) return;
  if (g == 0) sm_ml[slot * 16 + r16] = make_float2(m_run, o_l[0]);
  float* dst = sm_o + (slot * a.gqa + r16) * wave_row_floats<D>();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (SE % 4 == 0) {
#pragma unroll
      for (int dt = 0; dt < DT; dt += 4)
        *reinterpret_cast<f4_t*>(dst + o_slot(i, dt)) = f4_t{o[dt][i], o[dt + 1][i], o[dt + 2][i], o[dt + 3][i]};
    } else {
#pragma unroll
      for (int dt = 0; dt < DT; dt += 2)
        *reinterpret_cast<float2*>(dst + o_slot(i, dt)) = make_float2(o[dt][i], o[dt + 1][i]);
    }
  }
}


// ---------------------------------------------------------------------------
// Ranges.
// ---------------------------------------------------------------------------
// Position in the units laid end to end: unit (b, kvh) starts at position
// `start`, its `pages` pages of `len` tokens RangePlan::E positions later; its
// page ids begin at entry `row` of the CSR index.
struct Unit {
  int b, kvh, start, pages, len, row;
};

// The call's plan as every workgroup sees it: P positions in ranges of T.
struct RangePlan {
  int T, P, E;
  Unit first;  // the unit that holds position g * T (when g * T < P)
};

// Sequence b's page count, length and CSR row, read with scalar loads.
__device__ __forceinline__ void sequence_info(const Phase1Args& a, int b, int* pages, int* len, int* row) {
  if (a.csr) {
    const int r0 = min(max(load_uniform_i32(a.indptr + b), 0), a.max_pages);
    const int r1 = min(max(load_uniform_i32(a.indptr + b + 1), r0), a.max_pages);
    const int last = min(max(load_uniform_i32(a.lpl + b), 1), a.ps);
    *row = r0;
    *pages = r1 - r0;
    *len = *pages > 0 ? (*pages - 1) * a.ps + last : 0;
  } else {
    *len = max(load_uniform_i32(a.sl + (int64_t)b * a.ssl), 0);
    *pages = min(pages_for(a, *len), a.max_pages);
    *row = 0;
  }
}

// f(0), ..., f(N - 1), each with its index as a constant.
template <int N>
struct Index {
  static constexpr int value = N;
};
template <int N, class F>
__device__ __forceinline__ void each(F f) {
  if constexpr (N > 0) {
    each<N - 1>(f);
    f(Index<N - 1>());
  }
}

// 64 * NK sequences from b0 on, lane l holding b0 + l + 64k (a lane past the
// batch holds an empty one).
template <int NK>
struct Sequences {
  int pages[NK], len[NK], row[NK];
  __device__ __forceinline__ void load(const Phase1Args& a, int b0, int lane) {
    int w0[NK], w1[NK], w2[NK];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const int b = min(b0 + lane + 64 * k, a.batch - 1);
      w0[k] = a.csr ? a.indptr[b] : a.sl[(int64_t)b * a.ssl];
      w1[k] = a.csr ? a.indptr[b + 1] : 0;
      w2[k] = a.csr ? a.lpl[b] : 0;
    }
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const bool in = b0 + lane + 64 * k < a.batch;
      const int r = a.csr ? min(max(w0[k], 0), a.max_pages) : 0;
      const int csr_pages = min(max(w1[k], r), a.max_pages) - r;
      const int csr_len = csr_pages > 0 ? (csr_pages - 1) * a.ps + min(max(w2[k], 1), a.ps) : 0;
      const int l = max(w0[k], 0);
      const int n = a.csr ? csr_pages : min(pages_for(a, l), a.max_pages);
      row[k] = r;
      pages[k] = in ? n : 0;
      len[k] = in ? (a.csr ? csr_len : l) : 0;
    }
  }
};

// Plans the call from the sequence lengths.  Lengths of all sorts: each unit
// counts E = unit_extra positions at its front, T = ceil(P / G), at least
// min_chunk.  All the same page count: the units are cut alike, into as many
// pieces as ranges are left for each (E fills a unit up to whole ranges), or
// each range takes as many whole units - unless that leaves so much of the
// grid idle that the ranges are more than 1.6 times as long.  us cut alike /
// into equal ranges, by that ratio: 33 x 4096 of 32/8 heads (1.26) 88 / 92, 43
// (1.45) 113.8 / 114.9, 150 of 8/1 (1.58) 54.1 / 57.1, 72 of 32/8 (1.74) 208 /
// 194, 65 (1.92) 189 / 170, 129 (1.94) 367 / 325; 65 x 8192 at head_dim 64
// (1.92) 219 / 166.
// Empty sequences lie between units without a page; the workgroup whose range
// holds that position (the last range at the end) writes their zero rows:
// on_empty(b, owner) is called by the lane of every empty sequence b.  NK
// registers hold the table; a batch past 64 * NK is read twice in steps.
template <int NK, class F>
__device__ __forceinline__ RangePlan plan_ranges(const RangeArgs& a, int g, int lane, F on_empty) {
  Sequences<NK> s;
  const bool once = a.batch <= 64 * NK;
  int tot = 0, used = 0, most = 0, least = 0x7fffffff;
  for (int b0 = 0; b0 < a.batch; b0 += 64 * NK) {
    s.load(a, b0, lane);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      tot += s.pages[k];
      used += s.pages[k] > 0 ? 1 : 0;
      most = max(most, s.pages[k]);
      least = min(least, s.pages[k] > 0 ? s.pages[k] : 0x7fffffff);
    }
  }
  RangePlan p;
  tot = wave_sum_i32(tot);
  used = wave_sum_i32(used) * a.hkv;
  most = wave_max_i32(most);
  p.E = a.unit_extra;
  p.P = tot * a.hkv + used * p.E;
  p.T = max((p.P + a.groups - 1) / a.groups, max(a.min_chunk, 1));
  if (__builtin_amdgcn_ballot_w64(least < most) == 0 && used > 0) {
    int T, E = 0;
    if (used <= a.groups) {
      T = max((most + a.groups / used - 1) / (a.groups / used), a.min_chunk);
      E = (most + T - 1) / T * T - most;
    } else {
      T = (used + a.groups - 1) / a.groups * most;
    }
    if (5 * (int64_t)T <= 8 * (int64_t)p.T) {
      p.T = T;
      p.E = E;
      p.P = used * (most + E);
    }
  }
  const int lo = g * p.T;
  p.first = Unit{};
  int carry = 0;
  for (int b0 = 0; b0 < a.batch; b0 += 64 * NK) {
    if (!once) s.load(a, b0, lane);
    each<NK>([&](auto index) {
      constexpr int k = decltype(index)::value;
      const int x = s.pages[k] > 0 ? (s.pages[k] + p.E) * a.hkv : 0;
      const int incl = wave_incl_scan_i32(x, lane) + carry;
      const int excl = incl - x;
      const uint64_t hit = __builtin_amdgcn_ballot_w64(excl <= lo && lo < incl);
      if (hit != 0) {
        const int l = (int)__builtin_ctzll(hit);
        p.first.b = b0 + 64 * k + l;
        p.first.pages = __builtin_amdgcn_readlane(s.pages[k], l);
        p.first.len = __builtin_amdgcn_readlane(s.len[k], l);
        p.first.row = __builtin_amdgcn_readlane(s.row[k], l);
        const int seq0 = __builtin_amdgcn_readlane(excl, l);
        const int size = p.first.pages + p.E;
        p.first.kvh = __builtin_amdgcn_readfirstlane((lo - seq0) / size);
        p.first.start = seq0 + p.first.kvh * size;
      }
      const int b = b0 + lane + 64 * k;
      const bool empty = b < a.batch && s.pages[k] == 0;
      if (__builtin_amdgcn_ballot_w64(empty) != 0)
        on_empty(b, empty ? (p.P > 0 ? min(excl, p.P - 1) / p.T : 0) : -1);
      carry = __builtin_amdgcn_readlane(incl, 63);
    });
  }
  return p;
}

// The piece of unit u that the range [lo, hi) holds: pages [begin, end) of it
// (none if they are equal), one of n pieces, the first of them in range g1.
struct Piece {
  int begin, end, g1, n;
};
__device__ __forceinline__ Piece piece_of(const Unit& u, int E, int T, int lo, int hi) {
  const int page0 = u.start + E;
  const int begin = max(lo - page0, 0);
  const int g1 = (int)((uint32_t)page0 / (uint32_t)T);
  return Piece{begin, max(min(hi - page0, u.pages), begin), g1, (int)((uint32_t)(page0 + u.pages - 1) / (uint32_t)T) - g1 + 1};
}

// Work list of a range launch: the header of pa_decode.hip's lists, then one
// record of 32 int32 per workgroup: {b, head group, 2 unused, tokens, 2 unused,
// pages - 1, valid, CSR row, unit start, T, P, 1 if the workgroup writes zero
// rows, E, 1 unused, raw first page ids of the first segment's first 8 blocks
// (whole-page blocks), then sequences 2g and 2g + 1 of the batch as {pages,
// tokens, CSR row, owner of its zero rows or -1}}.
constexpr int kRlMagic = 0x574c4150;  // "PALW"

__device__ __forceinline__ const int32_t* list_sequence(const RangeArgs& a, int b) {
  return a.worklist + kRlHeaderInts + (int64_t)kRlRecordInts * (b >> 1) + 24 + 4 * (b & 1);
}

// Writes the zero rows of one sequence (all its query heads).
template <int D>
__device__ __forceinline__ void zero_sequence(const RangeArgs& a, int b, int threads) {
  const int total4 = a.rows * a.hkv * (D / 4);
  for (int e = threadIdx.x; e < total4; e += threads) {
    const int row = e / (D / 4);
    *reinterpret_cast<h4_t*>(a.out + (int64_t)b * a.sob + (int64_t)row * a.soh + (e - row * (D / 4)) * 4) = (h4_t)0;
  }
}

// The zero rows that a list leaves to workgroup g: lane l reads the owners of
// sequences l + 64k, all in one round trip.  (Reading them one after the other
// held up the workgroup that owns an empty sequence, and so the call: plan and
// run of 512 sequences of 8/1 heads, one of them empty, 143 us against 96.)
template <int D, int NK>
__device__ __forceinline__ void zero_listed(const RangeArgs& a, int g, int lane, int threads) {
  int owner[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) owner[k] = list_sequence(a, min(lane + 64 * k, a.batch - 1))[3];
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    uint64_t mine = __builtin_amdgcn_ballot_w64(lane + 64 * k < a.batch && owner[k] == g);
    for (; mine != 0; mine &= mine - 1) zero_sequence<D>(a, 64 * k + (int)__builtin_ctzll(mine), threads);
  }
}

template <int D, int NK>
__device__ __forceinline__ RangePlan plan_and_zero(const RangeArgs& a, int g, int lane, int threads) {
  return plan_ranges<NK>(a, g, lane, [&](int b, int owner) {
    uint64_t mine = __builtin_amdgcn_ballot_w64(owner == g);
    for (; mine != 0; mine &= mine - 1)
      zero_sequence<D>(a, __builtin_amdgcn_readlane(b, (int)__builtin_ctzll(mine)), threads);
  });
}

// Entry e of a unit whose first range is g1: its partial's slot.  Slot 2g + 1
// holds a unit's first piece (a workgroup has at most one unit that goes on
// past its range), slot 2g a later one (at most one that began before it).
__device__ __forceinline__ int entry_slot(int e) { return e == 0 ? 1 : 2 * e; }

// Folds `count` entries first, first + step, ... of a unit's partials, in entry
// order as MergeBatch does, for the group's (row, 4 columns) elements, and
// calls store(row, col, m, l, acc) for each.  Entries that a batch reads past
// the count lie past the unit's region (they read zeros) and fold with
// weight 0.  One workgroup folds a unit while the others have finished, so
// what counts is memory round trips: a thread with a second element loads
// N entries of both at once.
template <int D, int N, int X, class F>
__device__ __forceinline__ void fold_elements(__amdgpu_buffer_rsrc_t o_rsrc, __amdgpu_buffer_rsrc_t ml_rsrc, int first,
                                              int step, int count, int rows, int thread, int threads, F store) {
  for (int e0 = thread; e0 < rows * (D / 4); e0 += X * threads) {
    float m[X], l[X];
    f4_t acc[X];
#pragma unroll
    for (int x = 0; x < X; ++x) {
      m[x] = kNegInf;
      l[x] = 0.f;
      acc[x] = (f4_t)0.f;
    }
    for (int at = 0; at < count; at += N) {
      MergeBatch<N> p[X];
#pragma unroll
      for (int x = 0; x < X; ++x) {
        const int e = e0 + x * threads;
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const uint32_t r = (uint32_t)(entry_slot(first + (at + j) * step) * rows) + (uint32_t)(e / (D / 4));
          p[x].ml[j] = load_device_f2(ml_rsrc, r * 8u);
          p[x].o[j] = load_device_f4(o_rsrc, (r * (uint32_t)D + (uint32_t)(e % (D / 4)) * 4u) * 4u);
        }
      }
#pragma unroll
      for (int x = 0; x < X; ++x) p[x].fold(at, count, m[x], l[x], acc[x]);
    }
#pragma unroll
    for (int x = 0; x < X; ++x) {
      const int e = e0 + x * threads;
      if (e < rows * (D / 4)) store(e / (D / 4), e % (D / 4) * 4, m[x], l[x], acc[x]);
    }
  }
}

template <int D, class F>
__device__ __forceinline__ void fold_unit(__amdgpu_buffer_rsrc_t o_rsrc, __amdgpu_buffer_rsrc_t ml_rsrc, int first,
                                          int step, int count, int rows, int thread, int threads, F store) {
  if (rows * (D / 4) <= threads) {
    if (count <= 4)
      fold_elements<D, 4, 1>(o_rsrc, ml_rsrc, first, step, count, rows, thread, threads, store);
    else
      fold_elements<D, 8, 1>(o_rsrc, ml_rsrc, first, step, count, rows, thread, threads, store);
  } else {
    if (count <= 4)
      fold_elements<D, 4, 2>(o_rsrc, ml_rsrc, first, step, count, rows, thread, threads, store);
    else
      fold_elements<D, 8, 2>(o_rsrc, ml_rsrc, first, step, count, rows, thread, threads, store);
  }
}

// Merges the states of each kv head's nwl waves, threads over (row, 4
// consecutive head_dim slots), and writes unit u's output rows (final) or its
// piece's partial, with device-scope stores (coherent across the XCDs).
template <int D, int KVF>
__device__ __forceinline__ void write_piece(const RangeArgs& a, const Unit& u, int slot, bool final, int nwl, int thread,
                                            int threads, const float2* sm_ml, const float* sm_o) {
  const int rows = a.rows;
  _Float16* out_u = a.out + (int64_t)u.b * a.sob + (int64_t)(u.kvh * rows) * a.soh;
  const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(a.o_part + (int64_t)slot * rows * D, (uint32_t)(rows * D) * 4u);
  const __amdgpu_buffer_rsrc_t ml_rsrc = make_rsrc(a.ml_part + (int64_t)slot * rows, (uint32_t)rows * 8u);
  for (int e = thread; e < rows * (D / 4); e += threads) {
    const int row = e / (D / 4);
    const int col = (e - row * (D / 4)) * 4;
    const int head = (int)(((uint32_t)row * a.gqa_rcp) >> 16);  // in the group
    const int hrow = row - head * a.gqa;
    // Unrolled over the largest wave count, so all LDS reads issue together.
    float2 ml[kMaxWaves];
    f4_t ow[kMaxWaves];
#pragma unroll
    for (int w = 0; w < kMaxWaves; ++w) {
      if (w < nwl) {
        const int state = (w << a.nh_shift) + head;
        ml[w] = sm_ml[state * 16 + hrow];
        ow[w] = *reinterpret_cast<const f4_t*>(sm_o + (state * a.gqa + hrow) * wave_row_floats<D>() + col);
      }
    }
    float M = kNegInf;
#pragma unroll
    for (int w = 0; w < kMaxWaves; ++w)
      if (w < nwl) M = fmaxf(M, ml[w].x);
    f4_t acc = (f4_t)0.f;
    float Ls = 0.f;
#pragma unroll
    for (int w = 0; w < kMaxWaves; ++w) {
      if (w < nwl) {
        const float c = (ml[w].x == kNegInf) ? 0.f : exp2_fast(ml[w].x - M);
        Ls += c * ml[w].y;
        acc += c * ow[w];
      }
    }
    if (final) {
      const float inv = (kv_is_fp8<KVF>() ? a.v_fix : 1.f) / Ls;
      h4_t hv;
#pragma unroll
      for (int i = 0; i < 4; ++i) hv[i] = round16<KVF>(acc[i] * inv);
      *reinterpret_cast<h4_t*>(out_u + (int64_t)row * a.soh + col) = hv;
    } else {
      store_device(o_rsrc, (uint32_t)(row * D + col) * 4u, acc);
      if (col == 0) store_device(ml_rsrc, (uint32_t)row * 8u, make_float2(M, Ls));
    }
  }
}

// Workgroups of 8 waves for rows of at most 128 bytes, else 4 (the grid is one
// workgroup per CU): with 4, one wave per SIMD has the whole register file.
template <int D, int KVF>
constexpr int range_waves() { return D * kv_elem_bytes<KVF>() <= 128 ? 8 : 4; }

template <int D, int MODE, int KVF>
__global__ __launch_bounds__((range_waves<D, KVF>() * 64))
    __attribute__((amdgpu_waves_per_eu((range_waves<D, KVF>() / 4)))) void pad_range_kernel(const RangeArgs) {
  // The argument block is read afresh in each phase (the compiler cannot see
  // that the pointer is the same): kept in scalar registers across the
  // segment loop, its 60 words and the streaming loop's own would not fit
  // them, and the overflow went to vector registers and to scratch memory.
  auto kernarg = __builtin_amdgcn_kernarg_segment_ptr();
  auto args = [&]() -> const RangeArgs& {
    asm volatile("" : "+s"(kernarg));
    return *(const RangeArgs*)kernarg;
  };
  // Likewise the thread index: values that one phase forms from it must not
  // sit in vector registers across the others.
  auto thread = [&]() -> int {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  const RangeArgs& a = args();
  extern __shared__ float4 smem_f4[];
  const int nw = a.nw;
  float2* sm_ml = reinterpret_cast<float2*>(smem_f4);       // [nw][16]
  float* sm_o = reinterpret_cast<float*>(smem_f4) + nw * 32;  // [nw][gqa][D + 4]
  // [nw] K staging tiles, then (head_dim 256) one Q^T copy per kv head.
  char* k_stage_all = reinterpret_cast<char*>(sm_o + nw * a.gqa * wave_row_floats<D>());

  const int g = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int threads = nw * 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Waves 2^nh_shift apart share a kv head; wl is the wave's place among them.
  const int sub = wave & ((1 << a.nh_shift) - 1);
  const int wl = wave >> a.nh_shift;
  const int nwl = nw >> a.nh_shift;

  // The plan: from the work list when it carries this launch's key (every
  // length then comes from the list too, so all workgroups agree on it),
  // else from the sequence lengths.
  int T, P, E, phys_first = 0;
  Unit u;
  bool listed = false, first_known = false;
  if (a.worklist != nullptr) {
    const int32_t* r = a.worklist + kRlHeaderInts + (int64_t)kRlRecordInts * g;
    const int magic = load_uniform_i32(a.worklist);
    const int key = load_uniform_i32(a.worklist + 1);
    int f[15];
#pragma unroll
    for (int i = 0; i < 15; ++i) f[i] = load_uniform_i32(r + i);
    phys_first = load_uniform_i32(r + 16 + wl);
#pragma unroll
    for (int i = 0; i < 15; ++i) asm volatile("" : "+s"(f[i]));  // one round trip with the header
    asm volatile("" : "+s"(phys_first));
    listed = magic == kRlMagic && key == a.wl_key;
    if (listed) {
      T = f[11];
      P = f[12];
      E = f[14];
      u = Unit{f[0], f[1], f[10], f[7] + 1, f[4], f[9]};
      if (f[13] != 0) {
        if (a.batch <= 64)
          zero_listed<D, 1>(a, g, lane, threads);
        else
          zero_listed<D, kRangeMaxBatch / 64>(a, g, lane, threads);
      }
      // A record that does not describe ranges of this launch's shapes is
      // treated as none.
      if (f[8] == 0 || T <= 0 || E < 0 || u.b < 0 || u.b >= a.batch || u.kvh < 0 || u.kvh >= a.hkv || u.start < 0) return;
      first_known = true;
    }
  }
  if (!listed) {
    RangePlan p;
    if (a.batch <= 64)
      p = plan_and_zero<D, 1>(a, g, lane, threads);
    else
      p = plan_and_zero<D, 4>(a, g, lane, threads);
    T = p.T;
    P = p.P;
    E = p.E;
    u = p.first;
  }
  // Wave-uniform state stays in scalar registers (what came out of a wave
  // reduction or a division would sit in vector registers across the
  // streaming loop).
  auto scalar = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  T = scalar(T);
  E = scalar(E);
  const int lo = scalar(g * T);
  const int hi = scalar(min(lo + T, P));
  if (lo >= hi) return;

  // Pages, tokens and CSR row of sequence b: from the list, where the plan is.
  auto sequence = [&](const RangeArgs& a, int b, Unit& x) {
    if (listed) {
      const int32_t* s = list_sequence(a, b);
      x.pages = load_uniform_i32(s);
      x.len = load_uniform_i32(s + 1);
      x.row = load_uniform_i32(s + 2);
    } else {
      sequence_info(a, b, &x.pages, &x.len, &x.row);
    }
  };
  // Pieces of units that other ranges share: one that began before this range
  // and one that goes on past it.
  int n_pend = 0;
  int pend_unit[2] = {0, 0}, pend_n[2] = {0, 0}, pend_e[2] = {0, 0};
  for (;;) {
    const RangeArgs& a = args();
    u = Unit{scalar(u.b), scalar(u.kvh), scalar(u.start), scalar(u.pages), scalar(u.len), scalar(u.row)};
    // Bounds of every later read: the unit's pages lie in its row of the
    // index, and its ranges in the grid (a stale work list could say
    // otherwise).
    if (u.pages <= 0 || u.pages > a.max_pages || u.row < 0 || (a.csr && u.row > a.max_pages - u.pages)) return;
    const Piece piece = piece_of(u, E, T, lo, hi);
    const int p_begin = scalar(piece.begin), p_end = scalar(piece.end);
    const int g1 = scalar(piece.g1), n = scalar(piece.n);
    if (p_begin < p_end) {
      if (g < g1 || g1 + n > a.groups) return;
      const int32_t* ids_row = a.csr ? a.bt + u.row : a.bt + (int64_t)u.b * a.sbb;
      const int64_t ids_stride = a.csr ? 1 : a.sbp;
      if constexpr (MODE == kModeUniform) {
        if (!first_known) phys_first = first_page_id(a, ids_row, ids_stride, u.pages - 1, p_begin, wl);
      }
      const int t_begin = p_begin * a.ps;
      const int t_end = min(p_end * a.ps, u.len);
      const int nblk = scalar((t_end - t_begin + kBlockTokens - 1) / kBlockTokens);
      range_wave_loop<D, MODE, KVF>(a, phys_first, ids_row, ids_stride, u.b, (u.kvh << a.nh_shift) + sub, t_begin,
                                    t_end, nblk, wl, nwl, wave, thread() & 63, sm_ml, sm_o,
                                    k_stage_all + wave * k_stage_bytes<D>(),
                                    k_stage_all + (nw + sub) * k_stage_bytes<D>());
      __syncthreads();
      // A unit that lies inside this range is final.
      write_piece<D, KVF>(args(), u, 2 * g + (g == g1 ? 1 : 0), n == 1, nwl, thread(), threads, sm_ml, sm_o);
      if (n > 1) {
        const int i = g == g1 ? 1 : 0;
        pend_unit[i] = u.b * a.hkv + u.kvh;
        pend_n[i] = n;
        pend_e[i] = g - g1;
        n_pend |= 1 << i;
      }
      __syncthreads();  // the next segment's states overwrite the ones just read
    }
    first_known = false;
    u.start += u.pages + E;
    if (u.start >= hi) break;
    if (++u.kvh == a.hkv) {
      u.kvh = 0;
      do {  // empty sequences have no unit
        if (++u.b >= a.batch) return;
        sequence(a, u.b, u);
      } while (u.pages == 0);
    }
  }
  if (n_pend == 0) return;

  // Fold the shared units, as pa_decode.hip does: a workgroup counts itself in
  // once its partial stores have completed at device scope, and the last
  // one of a unit to arrive folds all its partials and resets the counter.
  // Past kTwoLevelSplits ranges, groups of 16 fold first.
  __shared__ int s_last[2];
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  {
    // Lane i counts piece i in: both arrivals are one round trip.
    const RangeArgs& a = args();
    const int i = thread();
    if (i < 2 && (n_pend >> i & 1) != 0) {
      const int n = i ? pend_n[1] : pend_n[0];
      const int mine = i ? pend_e[1] : pend_e[0];
      const bool grouped = n > kTwoLevelSplits;
      int* counter = grouped ? a.counters + (int64_t)a.batch * a.hkv + 2 * (g - mine) + (mine & ~15)
                             : a.counters + (i ? pend_unit[1] : pend_unit[0]);
      const int need = grouped ? min(16, n - (mine & ~15)) : n;
      s_last[i] = atomicAdd(counter, 1) == need - 1;
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int i = 0; i < 2; ++i) {
    const RangeArgs& a = args();
    if ((n_pend >> i & 1) == 0 || !s_last[i]) continue;
    const int unit = i ? pend_unit[1] : pend_unit[0];
    const int n = i ? pend_n[1] : pend_n[0];
    const int mine = i ? pend_e[1] : pend_e[0];
    const int base_slot = 2 * (g - mine);
    const int rows = a.rows;
    const uint32_t region_rows = (uint32_t)(2 * n - 1) * (uint32_t)rows;
    const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(a.o_part + (int64_t)base_slot * rows * D, region_rows * D * 4u);
    const __amdgpu_buffer_rsrc_t ml_rsrc = make_rsrc(a.ml_part + (int64_t)base_slot * rows, region_rows * 8u);
    int* unit_counter = a.counters + unit;
    int step = 1, count = n;
    if (n > kTwoLevelSplits) {
      const int grp0 = mine & ~15;
      const int gsize = min(16, n - grp0);
      int* group_counter = a.counters + (int64_t)a.batch * a.hkv + base_slot + grp0;
      fold_unit<D>(o_rsrc, ml_rsrc, grp0, 1, gsize, rows, thread(), threads,
                   [&](int row, int col, float m, float l, f4_t acc) {
                     store_device(o_rsrc, ((uint32_t)(entry_slot(grp0) * rows + row) * D + col) * 4u, acc);
                     // a row's (m, l) is read by every thread of the row: to LDS first
                     if (col == 0) sm_ml[row] = make_float2(m, l);
                   });
      __syncthreads();
      if (threadIdx.x < rows)
        store_device(ml_rsrc, (uint32_t)(entry_slot(grp0) * rows + threadIdx.x) * 8u, sm_ml[threadIdx.x]);
      if (threadIdx.x == 0) atomicExch(group_counter, 0);
      step = 16;
      count = (n + 15) >> 4;
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (threadIdx.x == 0) s_last[i] = atomicAdd(unit_counter, 1) == count - 1;
      __syncthreads();
      if (!s_last[i]) continue;
    }
    const int b = unit / a.hkv;
    const int kvh = unit - b * a.hkv;
    _Float16* out_u = a.out + (int64_t)b * a.sob + (int64_t)(kvh * rows) * a.soh;
    fold_unit<D>(o_rsrc, ml_rsrc, 0, step, count, rows, thread(), threads,
                 [&](int row, int col, float, float l, f4_t acc) {
                   const float inv = (kv_is_fp8<KVF>() ? a.v_fix : 1.f) / l;
                   h4_t hv;
#pragma unroll
                   for (int j = 0; j < 4; ++j) hv[j] = round16<KVF>(acc[j] * inv);
                   *reinterpret_cast<h4_t*>(out_u + (int64_t)row * a.soh + col) = hv;
                 });
    if (threadIdx.x == 0) atomicExch(unit_counter, 0);
  }
}

// Work-list planner: one wave per workgroup of the decode grid; lane i < 32
// writes word i of its record.
template <int NK>
__device__ __forceinline__ void write_record(const RangeArgs& a, int32_t* wl) {
  const int g = blockIdx.x;
  const int lane = threadIdx.x;
  uint64_t zeros = 0;
  int own[2] = {-1, -1};  // owners of sequences 2g, 2g + 1
  const RangePlan p = plan_ranges<NK>(a, g, lane, [&](int b, int owner) {
    zeros |= __builtin_amdgcn_ballot_w64(owner == g);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint64_t at = __builtin_amdgcn_ballot_w64(b == 2 * g + j);
      if (at != 0) own[j] = __builtin_amdgcn_readlane(owner, (int)__builtin_ctzll(at));
    }
  });
  const Unit& u = p.first;
  const int lo = g * p.T, hi = min(lo + p.T, p.P);
  const bool valid = lo < hi;
  const int begin = max(lo - u.start - p.E, 0);  // first page of the first segment
  int v = 0;
  switch (lane) {
    case 0: v = u.b; break;
    case 1: v = u.kvh; break;
    case 4: v = u.len; break;
    case 7: v = u.pages - 1; break;
    case 8: v = valid ? 1 : 0; break;
    case 9: v = u.row; break;
    case 10: v = u.start; break;
    case 11: v = p.T; break;
    case 12: v = p.P; break;
    case 14: v = p.E; break;
    default: break;
  }
  if (!valid) v = 0;
  if (lane == 13) v = zeros != 0 ? 1 : 0;
  if (lane >= 16 && lane < 24 && valid && a.ps % kBlockTokens == 0) {
    const int col = min(begin + block_page(a, lane - 16), u.pages - 1);
    v = a.csr ? a.bt[u.row + col] : a.bt[(int64_t)u.b * a.sbb + (int64_t)col * a.sbp];
  }
  int32_t* r = wl + kRlHeaderInts + (int64_t)kRlRecordInts * g;
  if (lane < 24) r[lane] = v;
  // Sequences 2g and 2g + 1, from the lanes and registers that hold them.
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int b = 2 * g + j;
    int pages = 0, len = 0, row = 0;
    if (b < a.batch) sequence_info(a, b, &pages, &len, &row);
    const int w = lane - 24 - 4 * j;
    if (w >= 0 && w < 4) r[lane] = w == 0 ? pages : (w == 1 ? len : (w == 2 ? row : own[j]));
  }
  if (g == 0 && lane < kRlHeaderInts)
    wl[lane] = lane == 0 ? kRlMagic : (lane == 1 ? a.wl_key : (lane == 2 ? a.groups : 0));
}

__global__ __launch_bounds__(64) void pad_range_plan_kernel(const RangeArgs a, int32_t* wl) {
  if (a.batch <= 64)
    write_record<1>(a, wl);
  else
    write_record<4>(a, wl);
}

hipError_t launch_range_plan(const RangeArgs& a, int32_t* wl, hipStream_t st) {
  hipLaunchKernelGGL(pad_range_plan_kernel, dim3(a.groups), dim3(64), 0, st, a, wl);
  return hipGetLastError();
}

template <int D, int MODE, int KVF>
static hipError_t launch_one(const RangeArgs& a, int nw, size_t lds, hipStream_t st) {
  hipLaunchKernelGGL((pad_range_kernel<D, MODE, KVF>), dim3(a.groups), dim3(nw * 64), lds, st, a);
  return hipGetLastError();
}

template <int D, int KVF>
static hipError_t launch_mode(const RangeArgs& a, int nw, size_t lds, hipStream_t st) {
  if (a.ps % kBlockTokens == 0) return launch_one<D, kModeUniform, KVF>(a, nw, lds, st);
  switch (a.ps) {
    case 1: return launch_one<D, kModeSubpage + 0, KVF>(a, nw, lds, st);
    case 2: return launch_one<D, kModeSubpage + 1, KVF>(a, nw, lds, st);
    case 4: return launch_one<D, kModeSubpage + 2, KVF>(a, nw, lds, st);
    case 8: return launch_one<D, kModeSubpage + 3, KVF>(a, nw, lds, st);
    default: return launch_one<D, kModeGeneric, KVF>(a, nw, lds, st);
  }
}

template <int KVF>
static hipError_t launch_dim(const RangeArgs& a, int head_dim, int nw, size_t lds, hipStream_t st) {
  switch (head_dim) {
    case 64: return launch_mode<64, KVF>(a, nw, lds, st);
    case 128: return launch_mode<128, KVF>(a, nw, lds, st);
    case 256: return launch_mode<256, KVF>(a, nw, lds, st);
    default: break;
  }
  if constexpr (!kv_is_fp8<KVF>()) {
    if (head_dim == 32) return launch_mode<32, KVF>(a, nw, lds, st);
    if (head_dim == 96) return launch_mode<96, KVF>(a, nw, lds, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_range(const RangeArgs& a, int head_dim, int kvf, int nw, size_t lds, hipStream_t st) {
  switch (kvf) {
    case kKvF16: return launch_dim<kKvF16>(a, head_dim, nw, lds, st);
    case kKvE4M3: return launch_dim<kKvE4M3>(a, head_dim, nw, lds, st);
    case kKvE5M2: return launch_dim<kKvE5M2>(a, head_dim, nw, lds, st);
    case kKvBF16: return launch_dim<kKvBF16>(a, head_dim, nw, lds, st);
    case kKvE4M3B: return launch_dim<kKvE4M3B>(a, head_dim, nw, lds, st);
    case kKvE5M2B: return launch_dim<kKvE5M2B>(a, head_dim, nw, lds, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pad
