// Stream decode for bf16 and fp8 pages on the bf16 matrix cores.
//
// The work partition, partial slots and segment records are those of the
// stream kernel (decode_stream_body): every wavefront takes an equal range of
// the flat page list, each unit's range leaves one partial, and
// decode_stream_merge_kernel combines them.  What differs is the page math.
// On the vector units a page costs 440-480 instructions (256 FMAs for the
// products of 4 query heads, the widening, the cross-lane score reduction),
// which takes longer than a reduced-precision page's bytes do.  Here both
// products run on the matrix cores and a page costs about 130 vector and 12
// matrix instructions.  64 sequences of 512-8192 tokens, 32/8 heads, one layer
// with its merge: fp8 pages 111 -> 70 us (347 MB, 4.9 TB/s), bf16 pages 125 ->
// 120 us (692 MB, 5.8 TB/s); a loads-only read of pages moves 6.6 TB/s, the
// launch's start, its end and the merge are the rest.
//
// Exactness.  A bf16 page value is exact in bf16, and so is the bare code
// value of an fp8 element (the key scale is part of qscale, the value scale
// multiplies the result).  The fp32 operand of each product (scaled query,
// probability) is split by truncation into three bf16 terms holding its 24
// significant bits.  The three terms of the G query heads are columns of one
// matrix operand, column 4 * term + head (8 * term + head and a second
// operand for the low terms at G = 8), so the split costs no extra matrix
// instructions: scores of the terms are added across columns, and the
// outputs' term columns are added once per unit.
//
// Pages go straight from global memory to LDS (global_load_lds, 1 KiB per
// instruction), two stages of one page per wavefront: no registers are held
// by loads in flight and no LDS store instruction is issued.  The 16-byte
// chunks of a row are XOR-swizzled by row through the lanes' source
// addresses, so that the operand reads hit distinct banks.  Keys are read as
// matrix operand A (16 keys x 32 dims) with 16-byte reads; values are
// transposed on the way out of LDS (ds_read_b64_tr_b16 / _b8), each lane
// getting the 4 keys of one dim whose probabilities the score tile left it.
//
// Shape, measured on the fp8 pages above (whole layer with the merge, us, at
// the time against 72 for this form): three wavefronts per SIMD 72, four 75-99
// (spills, and one more partial per wavefront for the merge; 80 now), two 73;
// a stage of two pages (whose P.V runs on the K = 32 instruction) with two
// wavefronts 77-80; three and four stages 76-80; a second query area, so that
// a unit's rows always come with its first page, 0-1 % less on units of a few
// pages and none here.  bf16 pages: two wavefronts per SIMD (LDS: 18 KB each)
// 120, one with two-page stages 123.
//
// The page descriptors (unit, physical page, visible tokens) of 64 pages are
// formed at once, one per lane, and read back with v_readlane: no scalar
// load or division stands between a page and the next one's loads.
//
// Special values.  The three terms of a finite operand times a finite element
// add up to their product, and a NaN or infinite operand is its high term with
// zeros beside it: fp8 pages, which hold no infinities, need nothing more.  A
// bf16 page's infinity times a term that is zero is a NaN that fp32 does not
// give.  Every such NaN reaches the range's sum or outputs, so a range of bf16
// pages that ends with a NaN there is scanned for infinities and, if it has
// one, computed again with fp32 arithmetic before it is published.  One layer
// of the 64 sequences above, one of them with a NaN element: bf16 pages 119 ->
// 122 us, fp8 pages 72 -> 73 (1100 and 730 when every such range was computed
// again, row by row); with an infinite key, bf16 pages 201 us.
#pragma once

#include "bf16.hpp"
#include "fp8.hpp"
#include "prefill_bmma.hpp"

namespace helix::hip {
namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
using prefill_detail::v4f;
using prefill_detail::v4s;
using prefill_detail::v8bf;
using prefill_detail::v8s;

constexpr int mma_waves_per_simd(int pf) { return pf == 1 ? 2 : 3; }

template <int G, int PF>
struct MmaGeom {
  static constexpr int kElem = PF == 1 ? 2 : 1;     // bytes per page element
  static constexpr int kRow = 128 * kElem;          // bytes per token row
  static constexpr int kPage = 16 * kRow;           // bytes of a K or V page
  static constexpr int kLoads = kPage / 1024;       // load instructions of a K or V page
  static constexpr int kStage = 2 * kPage;          // K page, then V page
  static constexpr int kStages = 2;
  static constexpr int kQuery = kStages * kStage;   // the unit's query rows
  static constexpr int kBytes = kQuery + G * 512;
};

// 16 bytes per lane from base + off to LDS byte address lds + 16 * lane,
// non-temporal (each page byte is read once per launch).
__device__ __forceinline__ void lds_stream16(const void* base, unsigned off, unsigned lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
               :
               : "v"(off), "s"(base), "{m0}"(lds)
               : "memory");
}

// Waits until at most n of this wavefront's loads are in flight (loads
// complete in order; the counts that occur are listed, others round down).
template <int USUAL>
__device__ __forceinline__ void wait_loads(int n) {
#define HELIX_WAIT(N) asm volatile("s_waitcnt vmcnt(" #N ")" ::: "memory")
  if (n == USUAL) {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(USUAL) : "memory");
  } else if (n >= 8) {
    if (n >= 12) HELIX_WAIT(12);
    else if (n >= 10) HELIX_WAIT(10);
    else if (n >= 9) HELIX_WAIT(9);
    else HELIX_WAIT(8);
  } else if (n >= 4) {
    if (n >= 6) HELIX_WAIT(6);
    else if (n >= 5) HELIX_WAIT(5);
    else HELIX_WAIT(4);
  } else {
    if (n >= 3) HELIX_WAIT(3);
    else if (n >= 2) HELIX_WAIT(2);
    else if (n >= 1) HELIX_WAIT(1);
    else HELIX_WAIT(0);
  }
#undef HELIX_WAIT
}

__device__ __forceinline__ const void* uniform_ptr(const void* p) {
  return reinterpret_cast<const void*>(
      uniform64(static_cast<long long>(reinterpret_cast<std::uintptr_t>(p))));
}

// Bits of term `term` of x's split (prefill_detail::split3: what remains of
// x after the higher terms, truncated to bf16; a non-finite x is its high
// term alone) in the low half, without branches: mask1 / mask2 are
// 0xffff0000 from the second / third term on, else 0.
__device__ __forceinline__ unsigned split_term(float x, unsigned mask1, unsigned mask2) {
  float t = x - __uint_as_float(__float_as_uint(x) & mask1);
  t -= __uint_as_float(__float_as_uint(t) & mask2);
  const bool drop = mask1 != 0u && !(fabsf(x) < INFINITY);
  return drop ? 0u : __float_as_uint(t) >> 16;
}

// Eight fp8 code values (two words) as one bf16 matrix operand.
__device__ __forceinline__ v8bf fp8_operand(unsigned w0, unsigned w1) {
  const uint2 a = prefill_detail::fp8_codes_bf16(w0);
  const uint2 b = prefill_detail::fp8_codes_bf16(w1);
  return __builtin_bit_cast(v8bf, make_uint4(a.x, a.y, b.x, b.y));
}

// Inclusive prefix sum over the wavefront of values whose total fits 31 bits
// (row shifts, then the row totals broadcast: six adds, no LDS exchanges).
__device__ __forceinline__ int wave_scan32(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31
  return v;
}
__device__ __forceinline__ long long wave_scan(int v, bool fits, int lane) {
  if (fits) return wave_scan32(v);
  long long incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const long long t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  return incl;
}

// A wavefront's range [g0, g1) of the flat page list (ranges of C pages) and
// the unit its first page belongs to; g0 >= g1: no pages.
struct MmaStart {
  long long g0, g1, C, unit_g;  // unit_g: flat index of the unit's first page
  int b, kvh, np, hist;
};
__device__ __forceinline__ MmaStart mma_start(const DecodeKernelArgs& a, int wave, int lane) {
  // 64 sums of a table row's pages fit 31 bits for any plausible table.
  const bool fits = a.max_blocks < (1 << 24);
  MmaStart st{};
  st.g0 = 1;
  long long per_head = 0;
  // The first 64 sequences' lengths and prefix sums stay in registers: a
  // batch of up to 64 reads its lengths once and is scanned once.
  int hist0 = -1, np0 = 0;
  long long incl0 = 0;
  for (int c0 = 0; c0 < a.batch; c0 += 64) {
    const int bb = c0 + lane;
    const int hist = bb < a.batch ? clamp_length(a.lengths[bb], a.max_blocks) : -1;
    const int np = bb < a.batch ? unit_pages(hist, a.first_page) : 0;
    const long long incl = wave_scan(np, fits, lane);
    if (c0 == 0) {
      hist0 = hist;
      np0 = np;
      incl0 = incl;
    }
    per_head += uniform64(__shfl(incl, 63, 64));
  }
  const long long total = per_head * a.kv_heads;
  st.C = uniform64((total + a.stream_waves - 1) / a.stream_waves);
  const long long g0 = uniform64(static_cast<long long>(wave) * st.C);
  if (g0 >= total) return st;
  st.g0 = g0;
  st.g1 = uniform64(g0 + st.C < total ? g0 + st.C : total);
  st.kvh = __builtin_amdgcn_readfirstlane(static_cast<int>(g0 / per_head));
  const long long rem = g0 - static_cast<long long>(st.kvh) * per_head;
  long long base = 0;
  for (int c0 = 0; c0 < a.batch; c0 += 64) {
    int hist = hist0, np = np0;
    long long incl = incl0;
    if (c0 != 0) {
      const int bb = c0 + lane;
      hist = bb < a.batch ? clamp_length(a.lengths[bb], a.max_blocks) : -1;
      np = bb < a.batch ? unit_pages(hist, a.first_page) : 0;
      incl = wave_scan(np, fits, lane);
    }
    const unsigned long long hit = __ballot(base + incl - np <= rem && rem < base + incl);
    if (hit != 0) {
      const int src = __ffsll(static_cast<long long>(hit)) - 1;
      st.b = __builtin_amdgcn_readfirstlane(c0 + src);
      st.np = __builtin_amdgcn_readlane(np, src);
      st.hist = __builtin_amdgcn_readlane(hist, src);
      st.unit_g = uniform64(g0 - (rem - (base + __shfl(incl - np, src, 64))));
      break;
    }
    base += uniform64(__shfl(incl, 63, 64));
  }
  return st;
}

// A page in flight, in scalar registers: its unit (kvh * batch + b), index in
// the unit, and flags.
struct PageInFlight {
  int unit, p, loads;  // loads: load instructions of the page itself
  unsigned meta;
};
constexpr unsigned kPageValid = 31u;    // visible tokens
constexpr unsigned kPageAny = 32u;
constexpr unsigned kPageFirst = 64u;    // the unit's first page in this wavefront's range
constexpr unsigned kPageEnd = 128u;     // its last
constexpr unsigned kPageTail = 256u;    // the unit's tail row
constexpr unsigned kPageBad = 512u;     // page or length outside the pool or table
constexpr unsigned kPageQuery = 1024u;  // its unit's query rows were loaded with it

template <int G, bool APPEND, int PF>
__device__ __forceinline__ void decode_mma_body(
    DecodeKernelArgs a, const std::uint32_t* __restrict__ tables,
    const std::int32_t* __restrict__ lengths, float* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int* __restrict__ segments,
    const std::int64_t* __restrict__ append_slots, int wave, int lane, unsigned char* lds) {
  a.tables = tables;
  a.lengths = lengths;
  a.out = out;
  a.part_o = part_o;
  a.part_ml = part_ml;
  a.segments = segments;
  a.append_slots = APPEND ? append_slots : nullptr;
  static_assert(PF == 1 || PF == 2, "bf16 or fp8 pages");
  constexpr int D = 128;
  constexpr int P = 16;
  constexpr bool FP8 = PF == 2;
  using Geo = MmaGeom<G, PF>;
  constexpr int HS = G == 8 ? 8 : 4;  // columns per term
  constexpr int NB = G == 8 ? 2 : 1;  // matrix operands of the three terms
  constexpr int kQueryLoads = (G * 32 + 63) / 64;

  const int col = lane & 15;
  const int grp = lane >> 4;
  const int head = col & (HS - 1);
  const int term = col / HS;
  // Bits a term's predecessors take off; columns that hold a term of a head.
  const unsigned mask1 = term >= 1 ? 0xffff0000u : 0u;
  const unsigned mask2 = G != 8 && term >= 2 ? 0xffff0000u : 0u;
  const unsigned used = term < 3 && head < G ? 0xffffu : 0u;
  const unsigned low_used = term == 0 ? 0xffffu : 0u;  // second operand (G = 8)
  const unsigned lds0 = prefill_detail::lds_address(lds);

  const MmaStart st = mma_start(a, wave, lane);
  if (st.g0 >= st.g1) return;
  const long long g0 = st.g0, g1 = st.g1, C = st.C;

  // Descriptors of up to 64 pages of the range, one per lane: pages
  // chunk_g + lane.  (ub, ukvh, unp, uhist) is the unit page `built` starts in
  // and `ubase` the flat index of its first page.
  int ub = st.b, ukvh = st.kvh, unp = st.np, uhist = st.hist;
  long long ubase = st.unit_g;
  int d_unit = 0, d_p = 0;
  unsigned d_meta = 0;
  long long d_off = 0;  // byte offset in a pool, or of the tail row in its tensor
  auto build = [&](long long gs) {
    const long long g = gs + lane;
    int b = 0, kvh = 0, p = 0, np = 1, hist = 0;
    bool in = false;
    const long long end = gs + 64 < g1 ? gs + 64 : g1;
    for (;;) {
      if (g >= ubase && g < ubase + unp && g < end) {
        in = true;
        b = ub;
        kvh = ukvh;
        p = static_cast<int>(g - ubase);
        np = unp;
        hist = uhist;
      }
      if (ubase + unp > end || ubase + unp >= g1) break;
      ubase += unp;
      if (++ub == a.batch) {
        ub = 0;
        ++ukvh;
      }
      ub = __builtin_amdgcn_readfirstlane(ub);
      ukvh = __builtin_amdgcn_readfirstlane(ukvh);
      uhist = clamp_length(prefill_detail::uniform_read(a.lengths + ub), a.max_blocks);
      unp = unit_pages(uhist, a.first_page);
      ubase = uniform64(ubase);
    }
    const bool tail = p == np - 1;
    d_unit = kvh * a.batch + b;
    d_p = p;
    unsigned meta = 0;
    if (in) {
      const int left = hist - (p + a.first_page) * P;
      meta = kPageAny | (tail ? 1u : static_cast<unsigned>(left < P ? left : P));
      if (p == 0 || g == g0) meta |= kPageFirst;
      if (tail || g + 1 == g1) meta |= kPageEnd;
      if (tail) meta |= kPageTail;
      if (hist < 0) meta |= kPageBad;
      std::uint32_t phys = 0;
      if (!tail) {
        phys = a.tables[static_cast<std::size_t>(b) * a.max_blocks + p + a.first_page];
        if (phys >= a.physical_blocks) {
          meta |= kPageBad;
          phys = 0;
        }
      }
      d_off = tail ? (static_cast<long long>(b) * a.kv_heads + kvh) * (D * 4)
                   : (static_cast<long long>(phys) * a.kv_heads + kvh) * Geo::kPage;
    }
    d_meta = meta;
    // No load of this is pending in the page loop.
    __builtin_amdgcn_s_waitcnt(0);
    if (in && p == 0) {
      // This wavefront holds the unit's first page: record which wavefronts
      // hold its partials for the merge.
      const unsigned rel = static_cast<unsigned>(g - g0) + static_cast<unsigned>(np - 1);
      const unsigned per_wave = C < 0x7fffffff ? static_cast<unsigned>(C) : 0x7fffffffu;
      reinterpret_cast<int2*>(a.segments)[d_unit] =
          make_int2(wave, static_cast<int>(rel / per_wave) + 1);
    }
  };

  // Source offset within a page of the 16 bytes lane `lane` brings with load
  // i: row and chunk of LDS position i * 1024 + lane * 16, chunk unswizzled.
  // Chunk c of row r sits at position c ^ swz(r): bf16 keys r, values
  // 2 (r & 7); fp8 keys r / 2, values r & 6.
  unsigned koff[Geo::kLoads], voff[Geo::kLoads];
#pragma unroll
  for (int i = 0; i < Geo::kLoads; ++i) {
    if constexpr (FP8) {
      const int r = 8 * i + (lane >> 3), pos = lane & 7;
      koff[i] = static_cast<unsigned>(r * Geo::kRow + ((pos ^ (r >> 1)) & 7) * 16);
      voff[i] = static_cast<unsigned>(r * Geo::kRow + (pos ^ (r & 6)) * 16);
    } else {
      const int r = 4 * i + (lane >> 4), pos = lane & 15;
      koff[i] = static_cast<unsigned>(r * Geo::kRow + (pos ^ r) * 16);
      voff[i] = static_cast<unsigned>(r * Geo::kRow + (pos ^ (2 * (r & 7))) * 16);
    }
  }

  // Rows that are not 16-byte aligned go through registers.
  auto copy_row = [&](const float* src, unsigned char* dst) {
    reinterpret_cast<float4*>(dst)[lane & 31] = make_float4(src[0], src[1], src[2], src[3]);
  };
  // Query rows of a unit into the query area.
  auto load_query_rows = [&](int unit) {
    const int b = unit % a.batch, kvh = unit / a.batch;
    const float* const rows = a.query + (static_cast<std::size_t>(b) * a.q_heads + kvh * G) * D;
    if (a.rows_aligned == 0) {
#pragma unroll 1
      for (int h = 0; h < G; ++h) {
        if (lane < 32) copy_row(rows + h * D + lane * 4, lds + Geo::kQuery + h * 512);
      }
      stream_sync<true>();
      return;
    }
    const void* q = uniform_ptr(rows);
#pragma unroll
    for (int i = 0; i < kQueryLoads; ++i) {
      if (G * 32 >= 64 || lane < G * 32) {
        lds_stream16(q, static_cast<unsigned>(i * 1024 + lane * 16), lds0 + Geo::kQuery + i * 1024);
      }
    }
  };

  long long next_g = g0;  // next page to load
  // Issues the loads of the next page into `stage`.  query_free: no page in
  // flight still needs the query area.
  auto issue = [&](int stage, bool query_free) -> PageInFlight {
    PageInFlight d{0, 0, 0, 0u};
    if (next_g >= g1) return d;
    const int i = static_cast<int>(next_g - g0) & 63;
    // The stage's last reads have returned before it is written again.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (i == 0) build(next_g);
    ++next_g;
    d.meta = __builtin_amdgcn_readlane(d_meta, i);
    d.unit = __builtin_amdgcn_readlane(d_unit, i);
    d.p = __builtin_amdgcn_readlane(d_p, i);
    const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(d_off), i);
    const unsigned hi = __builtin_amdgcn_readlane(
        static_cast<unsigned>(static_cast<unsigned long long>(d_off) >> 32), i);
    const std::size_t off = static_cast<std::size_t>(hi) << 32 | lo;
    const unsigned base = lds0 + static_cast<unsigned>(stage * Geo::kStage);
    if ((d.meta & kPageFirst) != 0 && query_free && a.rows_aligned != 0) {
      load_query_rows(d.unit);
      d.meta |= kPageQuery;
    }
    if ((d.meta & kPageTail) != 0) {
      // The tail's fp32 rows: lanes 0-31 the key, 32-63 the value.
      if (a.rows_aligned != 0) {
        const char* src = reinterpret_cast<const char*>(lane < 32 ? a.tail_key : a.tail_value);
        prefill_detail::lds_load16(src + off + (lane & 31) * 16, base);
        d.loads = 1;
      }
    } else {
      const char* kb = reinterpret_cast<const char*>(a.key_pool) + off;
      const char* vb = reinterpret_cast<const char*>(a.value_pool) + off;
#pragma unroll
      for (int j = 0; j < Geo::kLoads; ++j) lds_stream16(kb, koff[j], base + j * 1024);
#pragma unroll
      for (int j = 0; j < Geo::kLoads; ++j) lds_stream16(vb, voff[j], base + Geo::kPage + j * 1024);
      d.loads = 2 * Geo::kLoads;
    }
    return d;
  };

  v8s qop[NB][4];
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int s = 0; s < 4; ++s) qop[n][s] = v8s{0, 0, 0, 0, 0, 0, 0, 0};
  v4f acc[8];
  float m = -INFINITY, l = 0.0f;
  bool unit_bad = false;
  int unit_p = 0;  // first page of the unit in this wavefront's range

  // Dim of element j of matrix step s in group grp: the operand reads fetch
  // 16 bytes of a row, one step of bf16 or two of fp8.
  auto step_dim = [&](int s) { return FP8 ? 16 * (4 * (s >> 1) + grp) + 8 * (s & 1) : 32 * s + 8 * grp; };

  auto load_query = [&](const unsigned char* src) {
    const float* q = reinterpret_cast<const float*>(src) + head * D;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      float4 x0 = make_float4(0.f, 0.f, 0.f, 0.f), x1 = x0;
      if (head < G) {
        x0 = *reinterpret_cast<const float4*>(q + step_dim(s));
        x1 = *reinterpret_cast<const float4*>(q + step_dim(s) + 4);
      }
      const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = xs[j] * a.qscale;
        qop[0][s][j] = static_cast<short>(split_term(x, mask1, mask2) & used);
        if constexpr (G == 8) {
          qop[1][s][j] = static_cast<short>(split_term(x, ~0u << 16, ~0u << 16) & low_used);
        }
      }
    }
  };

  // The tail's fp32 rows onto the page grid, into row 0 of the stage's pages
  // (and, fused append, into the sequence's reserved page row).
  auto round_tail = [&](int b, int kvh, unsigned char* stage) {
    const float4 x = *reinterpret_cast<const float4*>(stage + lane * 16);
    const int j = lane & 31;
    const bool key = lane < 32;
    unsigned char* page = stage + (key ? 0 : Geo::kPage);
    long long dst = -1;
    if constexpr (APPEND) {
      const std::int64_t at = prefill_detail::uniform_read(a.append_slots + b);
      if (at >= 0) dst = ((at / P * static_cast<long long>(a.kv_heads) + kvh) * P + at % P) * D;
    }
    float* const pool = key ? a.append_key_pool : a.append_value_pool;
    if constexpr (FP8) {
      const unsigned w = fp8_pack4_scaled(x, key ? a.k_scale : a.v_scale);
      reinterpret_cast<unsigned*>(page)[j] = w;
      if (APPEND && dst >= 0) {
        reinterpret_cast<unsigned*>(reinterpret_cast<unsigned char*>(pool) + dst)[j] = w;
      }
    } else {
      const uint2 w = make_uint2(bf16_pack(x.x, x.y), bf16_pack(x.z, x.w));
      reinterpret_cast<uint2*>(page)[j] = w;
      if (APPEND && dst >= 0) {
        reinterpret_cast<uint2*>(reinterpret_cast<unsigned short*>(pool) + dst)[j] = w;
      }
    }
  };

  // Row of one head's result; its (m, l) beside a partial.
  auto result_row = [&](int b, int kvh, bool complete, int h) -> float* {
    if (complete) return a.out + (static_cast<std::size_t>(b) * a.q_heads + kvh * G + h) * D;
    const std::size_t unit = static_cast<std::size_t>(kvh) * a.batch + b;
    return a.part_o + ((unit + wave) * G + h) * D;
  };
  auto write_ml = [&](int b, int kvh, int h, float mh, float lh) {
    const std::size_t unit = static_cast<std::size_t>(kvh) * a.batch + b;
    a.part_ml[((unit + wave) * G + h) * 2] = mh;
    a.part_ml[((unit + wave) * G + h) * 2 + 1] = lh;
  };

  // The range [unit_p, last] of a bf16 unit again, in fp32 (Special values,
  // above): first a scan of its elements for infinities, then, if it has any,
  // the heads of a page together, the next page on its way meanwhile.  A lane
  // holds dims 32 (lane & 3) .. + 31 of key lane / 4 for the scores and dims
  // 2 lane, 2 lane + 1 of every value row.  `lds_q`: the finished page's
  // stage.  Returns false, with nothing written, if the range has no
  // infinity.
  auto redo = [&](int b, int kvh, int last, bool tailed, bool complete, unsigned char* lds_q) {
    const int hist = clamp_length(prefill_detail::uniform_read(a.lengths + b), a.max_blocks);
    const int pages = last - unit_p + (tailed ? 0 : 1);  // without the tail row
    const int first = unit_p + a.first_page;
    auto page_at = [&](int i) {  // byte offset of the i-th page in the pools
      const std::uint32_t phys = prefill_detail::uniform_read(
          a.tables + static_cast<std::size_t>(b) * a.max_blocks + first + i);
      return (static_cast<std::size_t>(phys) * a.kv_heads + kvh) * Geo::kPage;
    };
    const auto* const kpool = reinterpret_cast<const unsigned char*>(a.key_pool);
    const auto* const vpool = reinterpret_cast<const unsigned char*>(a.value_pool);
    // Two elements of the tail row on the page grid (rows at any 4-byte
    // address).
    const std::size_t tail_row = (static_cast<std::size_t>(b) * a.kv_heads + kvh) * D;
    auto rounded = [](const float* row) { return bf16_pack(row[0], row[1]); };

    // Smallest distance of any element (16 bits, sign off) from infinity.
    using Pair = unsigned short __attribute__((ext_vector_type(2)));
    Pair least = {0xffff, 0xffff};
    auto scan = [&](unsigned w) {
      least = __builtin_elementwise_min(
          least, __builtin_bit_cast(Pair, (w & 0x7fff7fffu) ^ 0x7f807f80u));
    };
    // (Rows past the history count too: that only costs the second pass.)
    constexpr int SP = G == 8 ? 1 : 2;  // pages at a time, as the registers allow
#pragma unroll 1
    for (int i = 0; i < pages; i += SP) {
      uint4 x[SP][2 * Geo::kLoads];
#pragma unroll
      for (int n = 0; n < SP; ++n) {
        const std::size_t off =
            page_at(min(i + n, pages - 1)) + static_cast<std::size_t>(lane) * 16;
#pragma unroll
        for (int j = 0; j < Geo::kLoads; ++j) {
          x[n][2 * j] = *reinterpret_cast<const uint4*>(kpool + off + j * 1024);
          x[n][2 * j + 1] = *reinterpret_cast<const uint4*>(vpool + off + j * 1024);
        }
      }
#pragma unroll
      for (int n = 0; n < SP * 2 * Geo::kLoads; ++n) {
        const uint4 w = x[n % SP][n / SP];
        scan(w.x), scan(w.y), scan(w.z), scan(w.w);
      }
    }
    if (tailed) {
      scan(rounded(a.tail_key + tail_row + 2 * lane));
      scan(rounded(a.tail_value + tail_row + 2 * lane));
    }
    if (__ballot(least[0] == 0 || least[1] == 0) == 0) return false;

    // Scaled query rows in LDS, 36 floats apart per 32 dims: the four lanes of
    // a key read distinct banks.
    const float* const rows = a.query + (static_cast<std::size_t>(b) * a.q_heads + kvh * G) * D;
    float* const q = reinterpret_cast<float*>(lds_q);
    for (int h = 0; h < G; ++h) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int d = lane + 64 * e;
        q[h * 144 + (d >> 5) * 36 + (d & 31)] = rows[h * D + d] * a.qscale;
      }
    }
    stream_sync<true>();
    const int steps = pages + (tailed ? 1 : 0);
    constexpr int HG = G < 4 ? G : 4;  // heads at a time, as the registers allow
#pragma unroll 1
    for (int h0 = 0; h0 < G; h0 += HG) {
      float o[HG][2], rm[HG], rl[HG];
#pragma unroll
      for (int h = 0; h < HG; ++h) {
        o[h][0] = o[h][1] = rl[h] = 0.0f;
        rm[h] = -INFINITY;
      }
      uint4 k[4];
      unsigned v[P];
      auto load_keys = [&](int i) {
        if (i < pages) {
          const unsigned char* const src = kpool + page_at(i) + lane * 64;
#pragma unroll
          for (int j = 0; j < 4; ++j) k[j] = *reinterpret_cast<const uint4*>(src + j * 16);
        } else {
          const float* const src = a.tail_key + tail_row + 32 * (lane & 3);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            k[j] = make_uint4(rounded(src + 8 * j), rounded(src + 8 * j + 2),
                              rounded(src + 8 * j + 4), rounded(src + 8 * j + 6));
          }
        }
      };
      auto load_values = [&](int i) {
        if (i < pages) {
          const unsigned char* const src = vpool + page_at(i) + lane * 4;
#pragma unroll
          for (int r = 0; r < P; ++r) {
            v[r] = *reinterpret_cast<const unsigned*>(src + r * Geo::kRow);
          }
        } else {
          v[0] = rounded(a.tail_value + tail_row + 2 * lane);
        }
      };
      load_keys(0);
      load_values(0);
#pragma unroll 1
      for (int i = 0; i < steps; ++i) {
        const int valid = i == pages ? 1 : min(P, hist - (first + i) * P);
        float s[HG];
#pragma unroll
        for (int h = 0; h < HG; ++h) {
          s[h] = 0.0f;
          const float* const qr = q + (h0 + h) * 144 + (lane & 3) * 36;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float4 x0 = *reinterpret_cast<const float4*>(qr + 8 * j);
            const float4 x1 = *reinterpret_cast<const float4*>(qr + 8 * j + 4);
            const float4 k0 = bf16_widen(k[j].x, k[j].y);
            const float4 k1 = bf16_widen(k[j].z, k[j].w);
            s[h] += x0.x * k0.x + x0.y * k0.y + x0.z * k0.z + x0.w * k0.w;
            s[h] += x1.x * k1.x + x1.y * k1.y + x1.z * k1.z + x1.w * k1.w;
          }
          s[h] += dpp<kDppQuadXor1>(s[h]);
          s[h] += dpp<kDppQuadXor2>(s[h]);
          // One head's query words in registers at a time.
          __builtin_amdgcn_sched_barrier(0);
        }
        if (i + 1 < steps) load_keys(i + 1);
        const bool seen = (lane >> 2) < valid;
#pragma unroll
        for (int h = 0; h < HG; ++h) {
          // (A key's four lanes hold the same bits.)
          float mn = seen ? s[h] : -INFINITY;
          mn = fmaxf(mn, dpp<kDppRowHalfMirror>(mn));
          mn = fmaxf(mn, dpp<kDppRowRor8>(mn));
          mn = fmaxf(prefill_detail::row_max(mn), rm[h]);
          const float alpha = exp2_ratio_raw(rm[h], mn);
          const float p = seen ? exp2_ratio_raw(s[h], mn) : 0.0f;
          float sum = p;
          sum += dpp<kDppRowHalfMirror>(sum);
          sum += dpp<kDppRowRor8>(sum);
          rl[h] = rl[h] * alpha + prefill_detail::row_sum(sum);
          rm[h] = mn;
          s[h] = p;
          o[h][0] *= alpha;
          o[h][1] *= alpha;
        }
#pragma unroll
        for (int r = 0; r < P; ++r) {
          if (r < valid) {
            const float v0 = __uint_as_float(v[r] << 16), v1 = __uint_as_float(v[r] & 0xffff0000u);
#pragma unroll
            for (int h = 0; h < HG; ++h) {
              const float p =
                  __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[h]), 4 * r));
              o[h][0] += p * v0;
              o[h][1] += p * v1;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (i + 1 < steps) load_values(i + 1);
      }
#pragma unroll
      for (int h = 0; h < HG; ++h) {
        const float sc = !complete ? 1.0f : rm[h] == -INFINITY ? NAN : 1.0f / rl[h];
        float* const row = result_row(b, kvh, complete, h0 + h) + 2 * lane;
        row[0] = o[h][0] * sc;
        row[1] = o[h][1] * sc;
        if (!complete && lane == 0) write_ml(b, kvh, h0 + h, rm[h], rl[h]);
      }
    }
    return true;
  };

  auto finalize = [&](const PageInFlight& d, unsigned char* stage) {
    const int b = d.unit % a.batch, kvh = d.unit / a.batch;
    const float lt = prefill_detail::row_sum(l);
    bool nan = !(lt < INFINITY);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = acc[dt][i];
        if constexpr (G == 8) {
          x += dpp<kDppRowRor8>(x);
        } else {
          x = term < 3 ? x : 0.0f;
          x += dpp<kDppRowRor8>(x);
          x += dpp<kDppRowRor4>(x);
        }
        acc[dt][i] = x;
        if constexpr (!FP8) nan = nan || isnan(x);
      }
    }
    const bool tailed = (d.meta & kPageTail) != 0;
    // With a cascade prefix every unit also has a prefix partial to merge.
    const bool complete = a.first_page == 0 && unit_p == 0 && tailed;
    if constexpr (!FP8) {
      if (!unit_bad && __ballot(nan && head < G) != 0) {
        const bool redone = redo(b, kvh, d.p, tailed, complete, stage);
        // Nothing of this path is pending afterwards: the compiler would
        // otherwise wait in the page loop for registers that are loaded here.
        __builtin_amdgcn_s_waitcnt(0);
        if (redone) return;
      }
    }
    float sc = FP8 ? a.v_scale : 1.0f;
    if (complete) sc = m == -INFINITY || unit_bad ? NAN : sc / lt;
    if (col < G) {
      // (The output, too, may lie at any 4-byte address.)
      using Row4 = float __attribute__((ext_vector_type(4), aligned(4)));
      Row4* row = reinterpret_cast<Row4*>(result_row(b, kvh, complete, col));
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        row[4 * dt + grp] = Row4{acc[dt][0] * sc, acc[dt][1] * sc, acc[dt][2] * sc,
                                 acc[dt][3] * sc};
      }
      if (!complete && grp == 0) write_ml(b, kvh, col, m, unit_bad ? NAN : lt);
    }
  };

  using LdsV4s = __attribute__((address_space(3))) v4s;
  using LdsV2i = __attribute__((address_space(3))) v2i;
  // This lane's operand reads within a stage.
  const unsigned k_at = static_cast<unsigned>(
      col * Geo::kRow + (FP8 ? ((grp ^ (col >> 1)) & 7) : (grp ^ col)) * 16);
  const int v_row = 4 * grp + (FP8 ? (col >> 1) & 3 : col >> 2);
  const unsigned v_at = static_cast<unsigned>(
      Geo::kPage + v_row * Geo::kRow +
      (FP8 ? (((col >> 3) ^ (v_row & 6)) * 16 + (col & 1) * 8)
           : ((2 * (v_row & 7)) * 16 + (col & 3) * 8)));

  // later: load instructions issued after the page's own.
  auto compute = [&](const PageInFlight& d, int stage, int later) {
    unsigned char* base = lds + stage * Geo::kStage;
    const int valid = static_cast<int>(d.meta & kPageValid);
    if ((d.meta & kPageFirst) != 0) {
      // The query rows were loaded ahead of the page: their split runs while
      // the page is still on its way.
      if ((d.meta & kPageQuery) == 0) {
        load_query_rows(d.unit);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      } else {
        wait_loads<2 * Geo::kLoads>(d.loads + later);
      }
      load_query(lds + Geo::kQuery);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) acc[dt] = v4f{0.f, 0.f, 0.f, 0.f};
      m = -INFINITY;
      l = 0.0f;
      unit_bad = false;
      unit_p = d.p;
    }
    wait_loads<2 * Geo::kLoads>(later);
    if ((d.meta & (kPageTail | kPageBad)) != 0) {
      unit_bad = unit_bad || (d.meta & kPageBad) != 0;
      if ((d.meta & kPageTail) != 0) {
        const int b = d.unit % a.batch, kvh = d.unit / a.batch;
        if (a.rows_aligned == 0) {
          const std::size_t row = (static_cast<std::size_t>(b) * a.kv_heads + kvh) * D;
          copy_row((lane < 32 ? a.tail_key : a.tail_value) + row + (lane & 31) * 4,
                   base + (lane < 32 ? 0 : 512));
          stream_sync<true>();
        }
        round_tail(b, kvh, base);
        stream_sync<true>();
      }
    }

    // Scores of all terms and heads; x[i] is key 4 grp + i.
    v4f s[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) s[n] = v4f{0.f, 0.f, 0.f, 0.f};
    if constexpr (FP8) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint4 w = *reinterpret_cast<const uint4*>(base + (k_at ^ (64 * u)));
        const v8bf k0 = fp8_operand(w.x, w.y);
        const v8bf k1 = fp8_operand(w.z, w.w);
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              k0, __builtin_bit_cast(v8bf, qop[n][2 * u]), s[n], 0, 0, 0);
          s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              k1, __builtin_bit_cast(v8bf, qop[n][2 * u + 1]), s[n], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const v8bf kk =
            __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4*>(base + (k_at ^ (64 * u))));
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              kk, __builtin_bit_cast(v8bf, qop[n][u]), s[n], 0, 0, 0);
        }
      }
    }
    float x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // Columns 8 apart first: each step then adds the same two numbers in
      // every column of a head, so all its columns hold the same bits (the
      // terms of one probability must come from one value).
      float v = s[0][i];
      if constexpr (G == 8) v += s[1][i];
      v += dpp<kDppRowRor8>(v);
      if constexpr (G != 8) v += dpp<kDppRowRor4>(v);
      x[i] = v;
    }
    const bool full = valid == P;
    if (!full) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (4 * grp + i >= valid) x[i] = -INFINITY;
      }
    }
    const float mx = prefill_detail::row_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
    const float mn = fmaxf(m, mx);
    if (__ballot(!(mn == m)) != 0) {  // some row's maximum moved
      const float alpha = exp2_ratio_raw(m, mn);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) acc[dt] *= alpha;
      l *= alpha;
      m = mn;
    }
    float pr[4];
    if (__ballot(!(fabsf(mn) < INFINITY)) == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) pr[i] = __builtin_amdgcn_exp2f(x[i] - mn);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) pr[i] = 4 * grp + i < valid ? exp2_ratio_raw(x[i], mn) : 0.0f;
    }
    l += (pr[0] + pr[1]) + (pr[2] + pr[3]);
    // This column's term of each probability (its bf16 truncation is the
    // packed high half).
    unsigned pw[2], pl[2];
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      unsigned r[2], q[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        float t = pr[i + e];
        t -= __uint_as_float(__float_as_uint(t) & mask1);
        if constexpr (G != 8) t -= __uint_as_float(__float_as_uint(t) & mask2);
        r[e] = __float_as_uint(t);
        if constexpr (G == 8) {
          // The low terms: columns 0-7 of the second operand.
          t = pr[i + e];
          t -= __uint_as_float(__float_as_uint(t) & 0xffff0000u);
          t -= __uint_as_float(__float_as_uint(t) & 0xffff0000u);
          q[e] = term == 0 ? __float_as_uint(t) : 0u;
        }
      }
      pw[i / 2] = __builtin_amdgcn_perm(r[1], r[0], 0x07060302u);
      if constexpr (G == 8) pl[i / 2] = __builtin_amdgcn_perm(q[1], q[0], 0x07060302u);
    }
    const v4s pop = __builtin_bit_cast(v4s, make_uint2(pw[0], pw[1]));
    const v4s plo = G == 8 ? __builtin_bit_cast(v4s, make_uint2(pl[0], pl[1])) : pop;
    // O^T += V^T P^T, 16 dims a tile: the lane's 4 keys (4 grp .. + 3) of
    // dim 16 dt + col against its own probabilities.
    auto add_tile = [&](int dt, uint2 w) {
      acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(v4s, w), pop, acc[dt],
                                                          0, 0, 0);
      if constexpr (G == 8) {
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(v4s, w), plo,
                                                            acc[dt], 0, 0, 0);
      }
    };
    // Rows past the visible tokens may hold anything: their keys' places in
    // the operand are cleared.
    const int seen = valid - 4 * grp;
    auto values = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      if constexpr (FP8) {
        const int keep = seen >= 4 ? ~0 : seen <= 0 ? 0 : (1 << (8 * seen)) - 1;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          // Lanes 0-7 of a group bring its 4 rows of tile 2 t, lanes 8-15 of
          // tile 2 t + 1, 8 bytes each; the transposed read returns 4 keys of
          // one dim of each.
          v2i w = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2i*)(base + (v_at ^ (32 * t))));
          if constexpr (!FULL) w &= keep;
          add_tile(2 * t, prefill_detail::fp8_codes_bf16(static_cast<unsigned>(w[0])));
          add_tile(2 * t + 1, prefill_detail::fp8_codes_bf16(static_cast<unsigned>(w[1])));
        }
      } else {
        const unsigned keep0 = (seen > 0 ? 0xffffu : 0u) | (seen > 1 ? 0xffff0000u : 0u);
        const unsigned keep1 = (seen > 2 ? 0xffffu : 0u) | (seen > 3 ? 0xffff0000u : 0u);
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          uint2 w = __builtin_bit_cast(
              uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4s*)(base + (v_at ^ (32 * dt)))));
          if constexpr (!FULL) w = make_uint2(w.x & keep0, w.y & keep1);
          add_tile(dt, w);
        }
      }
    };
    if (full) {
      values(std::true_type{});
    } else {
      values(std::false_type{});
    }
    if ((d.meta & kPageEnd) != 0) finalize(d, base);
  };

#pragma unroll
  for (int dt = 0; dt < 8; ++dt) acc[dt] = v4f{0.f, 0.f, 0.f, 0.f};
  PageInFlight now = issue(0, true);
  PageInFlight next = issue(1, (now.meta & kPageFirst) == 0);
  int stage = 0;
  while (now.meta != 0) {
    compute(now, stage, next.loads + ((next.meta & kPageQuery) != 0 ? kQueryLoads : 0));
    now = next;
    next = issue(stage, (now.meta & kPageFirst) == 0);
    stage ^= 1;
  }
}

}  // namespace
}  // namespace helix::hip
