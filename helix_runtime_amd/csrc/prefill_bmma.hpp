// Chunked-prefill attention for bf16 and fp8 pages on the bf16 matrix cores.
//
// The decomposition, masks, online softmax and special-value rules are those
// of prefill_body (one workgroup per (sequence, kv head) and 128 query rows,
// 16-row tiles, scores computed transposed so each lane holds keys of one
// query row).  What differs is the matrix
// arithmetic.  A bf16 page element is exact in bf16, and so is the bare code
// value of an fp8 element (the key scale joins the score scale and the value
// scale multiplies the output, as in the decode kernel).  The fp32 operand
// of each product (the scaled query, the probabilities) is split by
// truncation into three bf16 terms, hi + mid + lo, which hold its 24
// significant bits exactly.  Every product term is then exact in fp32, and
// three v_mfma_f32_16x16x32_bf16 replace each fp32 instruction (scores and
// P.V) at about five times the matrix throughput;
// only the order of the fp32 accumulation differs from the fp32 kernel.
//
// Special values.  A non-finite operand keeps only its hi term.  The split
// can only go wrong by giving NaN where fp32 does not: a zero term of one
// operand times an infinite element of the other (a query term against an
// infinite key, a probability of exactly 1 against an infinite value), and
// a value row that some row masks reaching that row (0 * inf).  Each such
// NaN reaches the row's accumulators or sum, so a work item whose rows end
// with a NaN there (or with a sum that is not finite) is flagged in
// redo[block], and the launcher runs
// prefill_body (fp32 operands, exact paths for these cases) over the
// flagged items only.  An item whose exact result is NaN anyway is just
// computed twice.
//
// Blocks of 32 keys (two pages) per LDS stage, so that both products run on
// the K = 32 instruction.  Scores come out as two 16-key tiles, keys
// 4 g + i and 16 + 4 g + i of row col in lane (g = lane / 16, col = lane %
// 16).  P.V contracts over the keys in any order, so its 32-key operand
// takes them in the order the scores left them: contraction index 8 g + j
// is key 4 g + j for j < 4 and key 16 + 4 g + j - 4 otherwise, and the V
// operand is read in that order.
//
// LDS: K and V rows as bf16 in key order, 256 bytes a row, their 16-byte
// chunks XOR-swizzled by row.  V is transposed on the way out
// (ds_read_b64_tr_b16: the 4 keys of one dim that a lane's score tile left
// it), so staging writes rows and bf16 pages need no staging code at all:
// they go from global memory to LDS directly.  Storing V transposed instead
// took four 2-byte LDS stores a thread and page, and every page went through
// registers.  16 sequences of 512 rows over 0-4096 tokens, 32/8 heads: bf16
// pages 965 -> 750 us, fp8 pages 1013 -> 805 us (their codes are widened
// once per workgroup on the way; widening them in the operand reads would
// repeat it in all eight wavefronts).
#pragma once

#include "prefill_body.hpp"

namespace helix::hip::prefill_detail {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v8s __attribute__((ext_vector_type(8)));

typedef short v4s __attribute__((ext_vector_type(4)));

constexpr int kBKeys = 2 * P;  // keys per LDS stage

struct PrefillBmmaShared {
  __align__(1024) unsigned short k[2][kBKeys * D];
  __align__(1024) unsigned short v[2][kBKeys * D];
  // The low bf16 term of each lane's query operand, [wave][step][lane]:
  // kept here rather than in registers, which the other two terms, the
  // accumulators and the staging fill.
  __align__(16) uint4 qlo[kRows / 16][4][64];
};

// Byte position in a stage of 16-byte chunk `chunk` of row `row` (keys 0 ..
// 31): chunks are XOR-swizzled by row, so that the operand reads (K: one
// chunk of 16 rows; V: one pair of chunks of 8 rows) hit distinct banks.
__device__ __forceinline__ unsigned bmma_k_at(int row, int chunk) {
  return static_cast<unsigned>(row * (2 * D) + ((chunk ^ row) & 15) * 16);
}
__device__ __forceinline__ unsigned bmma_v_at(int row, int chunk) {
  return static_cast<unsigned>(row * (2 * D) + (chunk ^ (2 * (row & 7))) * 16);
}

// A uniform read of memory that the kernel does not write, through the
// scalar cache.
template <typename T>
__device__ __forceinline__ T uniform_read(const T* p) {
  return *(const __attribute__((address_space(4))) T*)(reinterpret_cast<std::uintptr_t>(p));
}

// x = hi + mid + lo exactly (truncating splits of a finite fp32); a
// non-finite x is hi alone.  Results are bf16 bit patterns.  Range: lo's
// exponent is 16 or more below x's, so for |x| < 2^-109 lo can be a bf16
// subnormal, which the matrix cores may flush; mid likewise for |x| <
// 2^-117.  Then the terms sum to x within |x| * 2^-7 (an absolute error
// below 2^-116), far under any tolerance of the products they enter (the
// scaled query and the probabilities of a row whose sum is at least 1);
// such items are not flagged for the exact redo.
__device__ __forceinline__ void split3(float x, short& hi, short& mid, short& lo) {
  const unsigned u = __float_as_uint(x);
  hi = static_cast<short>(u >> 16);
  if (!isfinite(x)) {
    mid = 0;
    lo = 0;
    return;
  }
  const float r1 = x - __uint_as_float(u & 0xffff0000u);
  const unsigned u1 = __float_as_uint(r1);
  mid = static_cast<short>(u1 >> 16);
  const float r2 = r1 - __uint_as_float(u1 & 0xffff0000u);
  lo = static_cast<short>(__float_as_uint(r2) >> 16);
}

// split3 for a probability (in [0, 1], or NaN): no finiteness test.  For
// a finite p the terms are split3's.  A NaN p still gives a NaN middle term,
// so the row's accumulators end NaN as they must (the item is redone).
__device__ __forceinline__ void split3_prob(float x, short& hi, short& mid, short& lo) {
  const unsigned u = __float_as_uint(x);
  hi = static_cast<short>(u >> 16);
  const float r1 = x - __uint_as_float(u & 0xffff0000u);
  const unsigned u1 = __float_as_uint(r1);
  mid = static_cast<short>(u1 >> 16);
  const float r2 = r1 - __uint_as_float(u1 & 0xffff0000u);
  lo = static_cast<short>(__float_as_uint(r2) >> 16);
}

// Four fp8 code values (one word, lowest byte first) as four bf16 bit
// patterns, lowest first, two to a word.  Exact: every E4M3 value is a bf16
// value, and the scale is 1.
__device__ __forceinline__ uint2 fp8_codes_bf16(unsigned w) {
  const auto lo = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false);
  const auto hi = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true);
  return make_uint2(__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi));
}

__device__ __forceinline__ float bf16_bits_value(unsigned short h) {
  return __uint_as_float(static_cast<unsigned>(h) << 16);
}

// PF: 1 bf16 pages, 2 fp8 pages.  Standalone prefill only (no cascade).
// The workgroup has 8 wavefronts of 16 query rows each.
// redo[block] is written for every block: 1 when the item must be redone
// exactly.
template <int G, int PF>
__device__ __forceinline__ void prefill_body_bmma(PrefillKernelArgs a,
                                                  const std::uint32_t* __restrict__ tables,
                                                  const std::uint32_t* __restrict__ order,
                                                  std::uint32_t* __restrict__ redo,
                                                  std::uint32_t block, PrefillBmmaShared& sh) {
  static_assert(PF == 1 || PF == 2, "bf16 matrix-core prefill is for bf16 and fp8 pages");
  constexpr int PW = kRows / G;
  constexpr bool FP8 = PF == 2;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int col = lane & 15;
  const int grp = lane >> 4;

  std::uint32_t item = block;
  if (order != nullptr) {
    item = order[block];
  } else {
    const std::uint32_t x = item % a.pos_blocks;
    item = item - x + (a.pos_blocks - 1 - x);
  }
  const int pb = static_cast<int>(item % a.pos_blocks);
  const int kvh = static_cast<int>((item / a.pos_blocks) % a.kv_heads);
  const int b = static_cast<int>(item / a.pos_blocks / a.kv_heads);
  const int T = a.tokens;
  const int pos0 = pb * PW;

  int hist = __builtin_amdgcn_readfirstlane(a.lengths[b]);
  bool bad = hist < 0 || hist > a.max_blocks * P;
  if (bad) hist = 0;
  const int key_end = hist + min(T, pos0 + PW);
  const std::uint32_t* __restrict__ table = tables + static_cast<std::size_t>(b) * a.max_blocks;
  const std::size_t chunk_row0 = (static_cast<std::size_t>(b) * a.kv_heads + kvh) * T;
  // fp8: keys are bare code values, their scale joins the score scale.
  const float qs = FP8 ? a.qscale * a.k_scale : a.qscale;

  // Query operand: step s covers dims 32 s + 8 grp .. + 7 of row col (B operand
  // of S^T = K Q^T), as three bf16 terms.
  v8s qv[2][4];
  const int r = wave * 16 + col;
  const int head = kvh * G + r / PW;
  const int qpos = pos0 + r % PW;
  const bool valid = qpos < T;
  const std::size_t qrow = ((static_cast<std::size_t>(b) * a.q_heads + head) * T + qpos) * D;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    float4 x0 = make_float4(0.f, 0.f, 0.f, 0.f), x1 = x0;
    if (valid) {
      x0 = *reinterpret_cast<const float4*>(a.query + qrow + 32 * s + 8 * grp);
      x1 = *reinterpret_cast<const float4*>(a.query + qrow + 32 * s + 8 * grp + 4);
    }
    const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    v8s lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      short h, m, l;
      split3(xs[j] * qs, h, m, l);
      qv[0][s][j] = h;
      qv[1][s][j] = m;
      lo[j] = l;
    }
    sh.qlo[wave][s][lane] = __builtin_bit_cast(uint4, lo);
  }

  v4f o[8];  // O^T tiles: o[dt][i] = O[row col][dim 16 dt + 4 grp + i]
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = v4f{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  // Staging of a 16-key half (one page) of the next 32-key block.
  // - A bf16 page wholly in the history goes straight from global memory to
  //   LDS as stored: 4 wavefronts per half, each 1 KiB (4 rows) of the K page
  //   and of the V page.
  // - Everything else goes through registers: fp8 codes (widened on the way),
  //   chunk rows (rounded onto the page grid), zeros past the key range.
  //   Thread tid moves dims 4 scol .. + 3 of key row srow, the two halves one
  //   after the other, so only one page is held in registers.  The one bf16
  //   half where the history ends inside a page is loaded when it is stored,
  //   so that the loads of the others are of one kind (chunk rows).
  const int srow = tid >> 5;
  const int scol = tid & 31;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  auto direct = [&](int blk, int half) { return !FP8 && blk * kBKeys + half * P + P <= hist; };
  auto chunk_only = [&](int blk, int half) { return blk * kBKeys + half * P >= hist; };
  const int drow = 4 * (uwave & 3) + grp;  // row within the page
  const unsigned dk = bmma_k_at(drow, col), dv = bmma_v_at(drow, col);  // chunk at position col
  // Physical page of this wavefront's half of block blk (read a block ahead
  // of its loads).
  auto direct_page = [&](int blk) -> std::uint32_t {
    const int half = uwave >> 2;
    return direct(blk, half) ? uniform_read(table + blk * 2 + half) : 0u;
  };
  auto direct_load = [&](int buf, int blk, std::uint32_t page) {
    const int half = uwave >> 2;
    if (!direct(blk, half)) return;
    const unsigned at = static_cast<unsigned>(half * P * 2 * D + (uwave & 3) * 1024);
    // A page outside the pool is not read: zeros in its place.
    const bool ok = page < a.physical_blocks;
    bad = bad || !ok;
    const std::size_t off = (static_cast<std::size_t>(page) * a.kv_heads + kvh) * (P * D * 2);
    const auto* kb = ok ? reinterpret_cast<const unsigned char*>(a.key_pool) + off
                        : reinterpret_cast<const unsigned char*>(kZeroRows);
    const auto* vb = ok ? reinterpret_cast<const unsigned char*>(a.value_pool) + off
                        : reinterpret_cast<const unsigned char*>(kZeroRows);
    lds_load16_at(kb, ok ? dk : lane * 16u,
                  lds_address(reinterpret_cast<unsigned char*>(sh.k[buf]) + at));
    lds_load16_at(vb, ok ? dv : lane * 16u,
                  lds_address(reinterpret_cast<unsigned char*>(sh.v[buf]) + at));
  };
  const float* const chunk_k = a.chunk_key + chunk_row0 * D;
  const float* const chunk_v = a.chunk_value + chunk_row0 * D;
  float4 stk = make_float4(0.f, 0.f, 0.f, 0.f), stv = stk;
  auto stage_load = [&](int blk, int half) {
    const int pkey0 = blk * kBKeys + half * P;
    if constexpr (FP8) {
      const int key = pkey0 + srow;
      const bool in_hist = key < hist;
      std::size_t page_off = 0;
      bool page_ok = false;
      if (pkey0 < hist) {
        const std::uint32_t page = uniform_read(table + pkey0 / P);
        page_ok = page < a.physical_blocks;
        bad = bad || !page_ok;
        page_off = page_ok ? (static_cast<std::size_t>(page) * a.kv_heads + kvh) * P * D : 0;
      }
      stk = stv = make_float4(0.f, 0.f, 0.f, 0.f);
      if (in_hist) {
        if (page_ok) {  // the row's 4 codes in .x
          const std::size_t e = page_off + srow * D + scol * 4;
          stk.x = __uint_as_float(*reinterpret_cast<const unsigned*>(
              reinterpret_cast<const unsigned char*>(a.key_pool) + e));
          stv.x = __uint_as_float(*reinterpret_cast<const unsigned*>(
              reinterpret_cast<const unsigned char*>(a.value_pool) + e));
        }
      } else if (key < key_end) {
        const unsigned at = static_cast<unsigned>((key - hist) * D + scol * 4);
        stk = *reinterpret_cast<const float4*>(chunk_k + at);
        stv = *reinterpret_cast<const float4*>(chunk_v + at);
      }
    } else if (chunk_only(blk, half)) {
      // (A chunk's rows fit 32-bit offsets: 2^25 rows of one head are 16 GB.)
      const unsigned at =
          static_cast<unsigned>((min(pkey0 + srow, key_end - 1) - hist) * D + scol * 4);
      stk = *reinterpret_cast<const float4*>(chunk_k + at);
      stv = *reinterpret_cast<const float4*>(chunk_v + at);
    }
  };
  // Stores a staged half as bf16 rows (fp8: the bare code values).
  auto stage_store = [&](int buf, int blk, int half) {
    if (direct(blk, half)) return;
    const int kr = half * P + srow;
    const int key = blk * kBKeys + kr;
    uint2 kb, vb;  // 4 bf16 each, low half first
    auto rounded = [&](const float4& k, const float4& v) {
      if constexpr (FP8) {
        kb = fp8_codes_bf16(fp8_pack4_scaled(k, a.k_scale));
        vb = fp8_codes_bf16(fp8_pack4_scaled(v, a.v_scale));
      } else {
        kb = make_uint2(bf16_pack(k.x, k.y), bf16_pack(k.z, k.w));
        vb = make_uint2(bf16_pack(v.x, v.y), bf16_pack(v.z, v.w));
      }
    };
    if constexpr (FP8) {
      if (key < hist) {
        kb = fp8_codes_bf16(__float_as_uint(stk.x));
        vb = fp8_codes_bf16(__float_as_uint(stv.x));
      } else {
        rounded(stk, stv);
      }
    } else if (chunk_only(blk, half)) {
      rounded(stk, stv);
      if (key >= key_end) kb = vb = make_uint2(0u, 0u);
    } else {
      const int pkey0 = blk * kBKeys + half * P;
      const std::uint32_t page = uniform_read(table + pkey0 / P);
      const bool ok = page < a.physical_blocks;
      bad = bad || !ok;
      kb = vb = make_uint2(0u, 0u);
      if (key < hist) {
        if (ok) {
          const std::size_t e =
              (static_cast<std::size_t>(page) * a.kv_heads + kvh) * P * D + srow * D + scol * 4;
          kb = *reinterpret_cast<const uint2*>(
              reinterpret_cast<const unsigned short*>(a.key_pool) + e);
          vb = *reinterpret_cast<const uint2*>(
              reinterpret_cast<const unsigned short*>(a.value_pool) + e);
        }
      } else if (key < key_end) {
        const unsigned at = static_cast<unsigned>((key - hist) * D + scol * 4);
        rounded(*reinterpret_cast<const float4*>(chunk_k + at),
                *reinterpret_cast<const float4*>(chunk_v + at));
      }
    }
    const unsigned part = static_cast<unsigned>((scol & 1) * 8);
    *reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(sh.k[buf]) +
                              bmma_k_at(kr, scol >> 1) + part) = kb;
    *reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(sh.v[buf]) +
                              bmma_v_at(kr, scol >> 1) + part) = vb;
  };

  __shared__ int s_redo;
  if (tid == 0) s_redo = 0;  // published by the first barrier below
  const int nblocks = (key_end + kBKeys - 1) / kBKeys;
  auto block_barrier = [&]() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  std::uint32_t page_ahead = 0;
  if (nblocks > 0) {
    direct_load(0, 0, direct_page(0));
    page_ahead = direct_page(1);
    stage_load(0, 0);
    stage_store(0, 0, 0);
    stage_load(0, 1);
    stage_store(0, 0, 1);
  }
  block_barrier();
  // Operand reads: K row 16 h + col, chunk 4 s + grp; V rows 4 grp .. + 3 of
  // a page, 16 dims of tile dt, transposed on the way out of LDS.
  const unsigned kop_at = bmma_k_at(col, grp);
  const int vrow = 4 * grp + (col >> 2);
  const unsigned vop_at = bmma_v_at(vrow, 0) + static_cast<unsigned>((col & 3) * 8);
  for (int n = 0; n < nblocks; ++n) {
    const int buf = n & 1;
    const bool next = n + 1 < nblocks;
    if (next) {
      direct_load(buf ^ 1, n + 1, page_ahead);
      page_ahead = direct_page(n + 2);
      stage_load(n + 1, 0);
    }
    const unsigned char* K = reinterpret_cast<const unsigned char*>(sh.k[buf]);
    const unsigned char* V = reinterpret_cast<const unsigned char*>(sh.v[buf]);

    // S^T = K Q^T on the bf16 matrix cores: st[h] holds keys
    // 16 h + 4 grp + i of query row col.
    v4f st[2];
    st[0] = st[1] = v4f{0.f, 0.f, 0.f, 0.f};
    // Raised wave priority over the matrix instructions: the waves of one
    // workgroup reach them together (barriers), and the softmax and staging
    // of the other workgroup on the CU fill the gaps.
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const v8bf qlo = __builtin_bit_cast(v8bf, sh.qlo[wave][s][lane]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v8bf kop = __builtin_bit_cast(
            v8bf, *reinterpret_cast<const v8s*>(K + h * (P * 2 * D) + (kop_at ^ (64u * s))));
        st[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop, qlo, st[h], 0, 0, 0);
#pragma unroll
        for (int term = 1; term >= 0; --term) {
          st[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              kop, __builtin_bit_cast(v8bf, qv[term][s]), st[h], 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_s_setprio(0);
    float p[8];  // p[4 h + i]: key 16 h + 4 grp + i
    const bool full = (n + 1) * kBKeys <= min(key_end, hist + pos0 + 1);
    auto softmax = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      float x[8];
      bool vis[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = n * kBKeys + 16 * (j >> 2) + 4 * grp + (j & 3);
        vis[j] = FULL || (key < key_end && (key < hist || key - hist <= qpos));
        x[j] = vis[j] ? st[j >> 2][j & 3] : -INFINITY;
      }
      const float mx = row_max(fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                                     fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7]))));
      const float mn = fmaxf(m, mx);
      // Branch-free rescale (alpha is 1 for rows whose maximum held).
      const float alpha = exp2_ratio(m, mn);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) o[dt] *= alpha;
      if (FULL && __ballot(!(fabsf(mn) < INFINITY)) == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = __builtin_amdgcn_exp2f(x[j] - mn);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = vis[j] ? exp2_ratio(x[j], mn) : 0.f;
      }
      // The lane's own keys; the row's four lanes are added at the end.
      l = l * alpha + (((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])));
      m = mn;
    };
    if (full) {
      softmax(std::true_type{});
    } else {
      softmax(std::false_type{});
    }

    if (next) {
      stage_store(buf ^ 1, n + 1, 0);
      stage_load(n + 1, 1);
    }

    {
      // O^T += V^T P^T: A = V^T rows (dims 16 dt + col) at contraction
      // indices 8 grp .. + 7, B = the lane's own 8 probabilities of row col
      // in the same order, as three bf16 terms.
      v8s pv[3];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        short h, mm, lo;
        split3_prob(p[j], h, mm, lo);
        pv[0][j] = h;
        pv[1][j] = mm;
        pv[2][j] = lo;
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        using LdsV4s = __attribute__((address_space(3))) v4s;
        const unsigned char* vp = V + (vop_at ^ (32u * dt));
        const v4s v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4s*)(vp));
        const v4s v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4s*)(vp + P * 2 * D));
        const v8bf vop = __builtin_bit_cast(
            v8bf, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int term = 2; term >= 0; --term) {
          o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vop, __builtin_bit_cast(v8bf, pv[term]), o[dt], 0, 0, 0);
        }
      }
    }

    __builtin_amdgcn_s_setprio(0);
    if (next) stage_store(buf ^ 1, n + 1, 1);
    block_barrier();
  }

  bool nan_row = false;
  l = row_sum(l);
  nan_row = nan_row || !(l < INFINITY);  // NaN, or a sum that overflowed
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) nan_row = nan_row || isnan(o[dt][i]);
  if (__ballot(nan_row) != 0 && lane == 0) s_redo = 1;
  const int any_bad = __syncthreads_or(bad);
  if (tid == 0) redo[block] = s_redo != 0 ? 1u : 0u;
  const float vscale = FP8 ? a.v_scale : 1.0f;
  if (qpos >= T) return;
  const bool no_result = any_bad || m == -INFINITY;
  const float inv = no_result ? NAN : vscale / l;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    float4 r = make_float4(o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
    if (no_result) r = make_float4(NAN, NAN, NAN, NAN);
    *reinterpret_cast<float4*>(a.out + qrow + 16 * dt + 4 * grp) = r;
  }
}

}  // namespace helix::hip::prefill_detail
