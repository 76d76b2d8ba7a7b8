// Sparse flash attention forward at D = 512 for few heads (up to 32 per
// workgroup): the heads of a tensor-parallel shard.
//
// A row's tokens cost the same gather (1152 bytes each) whatever the number
// of heads, and below about 64 heads that gather, not the matrix cores, is the
// bound: 32 tokens are 36 KB, 640 cycles of a CU at the 56 bytes per clock
// that whole-row loads reach from L2, against 17 MFMAs (270 cycles) per head
// tile.  The kernels of sfa_fwd.hip run every row on 64- or 128-head
// workgroups of eight waves with two workgroup barriers per 32-token tile; at
// 32 heads three quarters of their MFMAs multiplied zeros and a tile still
// took 4.2 k cycles.  Measured (one MI355X, through the Python API): 8192
// causal rows of 2048 tokens, 16 / 32 heads 3.87 / 3.89 -> 1.24 / 1.43 ms; a
// packed batch of 5247 rows of up to 1024 tokens, 32 heads 1.34 -> 0.44 ms
// (10 TB/s of gathered rows; the same loop without the softmax, on rows that
// stay in L2, reaches 15.5).  The 32-head kernels spill 2 to 19 registers (12 to
// 80 bytes of scratch per lane; 36 to 74, 116 to 188 bytes, with the 64-bit
// gather), none of them inside the tile loop.
//
// Here every wave works alone: it takes its own range of index positions,
// compacts them, gathers 16-token tiles by LDS-DMA into its own two-buffer
// ring and runs both products on them for all heads of the workgroup, with no
// barrier in the loop, so the four waves of a CU drift apart and one wave's
// products and softmax run while another's gather is issued.
//  * S^T = K . Q^T on 16x16x32 (one K fragment read serves HT head tiles).
//  * At 32 heads O^T += V^T . P^T runs on 32x32x16: the C layout of S^T becomes
//    its B layout by two v_permlane16_swap of the packed numerators (no LDS);
//    at 16 heads on 16x16x16, whose B layout is the C layout of S^T.
//  * The reference max of a head is that of the row's first 32 tokens (two
//    tiles, scored once before the loop), as in sfa_fwd.hip, and one for all
//    waves of a row: the numerators round as they do there, and a large score
//    at the start of a row is every wave's reference.  Scores that pass it by
//    more than kRefSlack (log2 units) send the wave through its positions a
//    second time with the exact maxima.
//  * TW = 1 (many rows: prefill): one wave per workgroup and row, four
//    workgroups per CU.  TW = 4 (fewer rows than wave slots): a row's positions
//    are dealt to four waves, whose (O, max, sum) are merged in fp32 through
//    the idle rings at the end.  Launches that split a row's tokens over
//    workgroups (decode) run the 64-head kernel of sfa_fwd.hip: with a few
//    tiles per wave the start of four independent waves and their merge cost
//    more than the padding (32 rows of 16 heads: 27.4 against 24.3 us).
#include <type_traits>

#include "sfa_fwd.h"

namespace dsa {

namespace {

constexpr int kFewD = 512;
constexpr int kFewTile = 16;
constexpr int kFewChunk = 512;  // positions compacted at a time (8 per lane)

// zero row for -1 pages and padding on the 64-bit gather path
__device__ __attribute__((aligned(16))) unsigned char g_few_zero_row[1024];

// 16 bytes per lane into LDS at lds + 16 lane, from voff + 256 q
__device__ __forceinline__ void few_dma_buf(unsigned lds, int q, int voff, __amdgpu_buffer_rsrc_t rsrc) {
  const unsigned m = lds - q * 256;
  if (q == 0) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(m), "v"(voff), "s"(rsrc) : "memory");
  if (q == 1) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen offset:256 lds" :: "s"(m), "v"(voff), "s"(rsrc) : "memory");
  if (q == 2) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen offset:512 lds" :: "s"(m), "v"(voff), "s"(rsrc) : "memory");
  if (q == 3) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen offset:768 lds" :: "s"(m), "v"(voff), "s"(rsrc) : "memory");
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T, int HT, int TW, bool BUF>
__global__ __launch_bounds__(TW * 64, 1) void sfa_fwd_few_kernel(SfaFwdParams p) {
  using E = Elem<T>;
  using V8 = typename E::v8;
  typedef T T4 __attribute__((ext_vector_type(4)));
  static_assert(HT == 1 || HT == 2, "heads");
  constexpr bool kSplitP = __is_same(T, bf16);
  constexpr int D = kFewD, DR = 64, TILE = kFewTile;
  constexpr int HEADS = HT * 16;
  constexpr int KS = (D + DR) / 32, KSN = D / 32;
  constexpr int NOPE = TILE * D * 2;            // bytes of a tile's nope rows
  constexpr int BUFB = NOPE + TILE * DR * 2;    // and with its rope rows
  constexpr int NDMA = TILE + TILE / 8;         // 1 KB DMAs per tile: a nope row, or eight rope rows
  constexpr int LIST = kFewChunk + TILE;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[TW][2 * BUFB];
  __shared__ int s_list[TW][LIST];
  __shared__ float s_st[TW > 1 ? TW : 1][3][HEADS];
  __shared__ float s_ref[TW][HEADS];
  __shared__ int s_cnt[TW], s_tiles[TW];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;

  const int64_t row = sfa_block_row(p, (int)(blockIdx.x & 7), (int)(blockIdx.x >> 3));  // n1 <= HEADS
  if (row < 0) return;

  // ---- this wave's positions ----
  const RowInfo ri = sfa_row_info(p, (int)row);
  const int32_t* idx_row = p.idx + row * p.K;
  const int total_pos = p.K * p.bs;
  const int per_wave = (total_pos + TW - 1) / TW;
  const int p0 = wave * per_wave, p1 = min(total_pos, p0 + per_wave);
  constexpr int RPL = kFewChunk / 64;
  int ids[RPL];
  auto load_ids = [&](int c) {
#pragma unroll
    for (int u = 0; u < RPL; ++u) {
      const int pos = c + u * 64 + lane;
      ids[u] = pos < p1 ? sfa_load_id(p, idx_row, pos) : -1;
    }
  };
  load_ids(p0);
  asm volatile("" ::: "memory");  // the index entries go out before Q

  // ---- Q (B operand of S^T): lane -> head li of each head tile, k = 8 lg .. ----
  V8 qf[HT][KS];
  const u32x4 z4 = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int ht = 0; ht < HT; ++ht) {
    const int head = ht * 16 + li;
    const bool hv = head < p.n1;
    const int64_t hs = row * p.n1 + (hv ? head : 0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 v = ks < KSN ? *(const u32x4*)((const T*)p.q + hs * D + ks * 32 + lg * 8)
                               : *(const u32x4*)((const T*)p.qr + hs * DR + (ks - KSN) * 32 + lg * 8);
      qf[ht][ks] = as_v8<V8>(hv ? v : z4);
    }
  }

  // ---- gather ----
  int* const list = s_list[wave];
  unsigned char* const ring = smem[wave];
  const unsigned ring_base = (unsigned)(uintptr_t)ring;
  __amdgpu_buffer_rsrc_t rk, rr;
  if constexpr (BUF) {
    rk = __builtin_amdgcn_make_buffer_rsrc((void*)p.k, (short)0, (int)(p.kv_rows * D * 2), 0x00020000);
    rr = __builtin_amdgcn_make_buffer_rsrc((void*)p.kr, (short)0, (int)(p.kv_rows * DR * 2), 0x00020000);
  }
  // A buffer holds its 16 nope rows in four column quarters of 4 KB (row r of
  // a quarter: 256 bytes, 16-byte chunk c at c ^ nope_swz(r)), then the rope
  // rows (chunk c at c ^ rope_swz(r)).  One DMA moves a quarter of four rows
  // or eight rope rows; the quarter moves the global and the LDS address
  // alike, so it is the instruction's offset and M0 the rest.
  struct Rows { int nope[4], rope[2]; };
  auto rows_of = [&](int t) -> Rows {
    int ln = lane;
    asm volatile("" : "+v"(ln));  // the chunk offsets are recomputed per tile, not held in registers
    Rows r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r.nope[j] = list[t * TILE + j * 4 + (ln >> 4)];
#pragma unroll
    for (int j = 0; j < 2; ++j) r.rope[j] = list[t * TILE + j * 8 + (ln >> 3)];
    if constexpr (BUF) {
      // byte offsets; a row of -1 (a missing page, padding) is out of range and reads zeros
#pragma unroll
      for (int j = 0; j < 4; ++j)
        r.nope[j] = r.nope[j] >= 0 ? r.nope[j] * (D * 2) + ((ln & 15) ^ nope_swz(j * 4 + (ln >> 4))) * 16 : (int)0x80000000;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        r.rope[j] = r.rope[j] >= 0 ? r.rope[j] * (DR * 2) + ((ln & 7) ^ rope_swz(j * 8 + (ln >> 3))) * 16 : (int)0x80000000;
    }
    return r;
  };
  auto issue_nope = [&](const Rows& r, int b, int q, int j) {
    const unsigned dst = ring_base + b * BUFB + q * 4096 + j * 1024;
    if constexpr (BUF) {
      few_dma_buf(dst, q, r.nope[j], rk);
    } else {
      const int off = ((lane & 15) ^ nope_swz(j * 4 + (lane >> 4))) * 16 + q * 256;
      dma_glb16(dst, (r.nope[j] >= 0 ? (const unsigned char*)p.k + (int64_t)r.nope[j] * (D * 2) : g_few_zero_row) + off);
    }
  };
  auto issue_rope = [&](const Rows& r, int b, int j) {
    const unsigned dst = ring_base + b * BUFB + NOPE + j * 1024;
    if constexpr (BUF) {
      dma_buf16(dst, r.rope[j], rr);
    } else {
      const int off = ((lane & 7) ^ rope_swz(j * 8 + (lane >> 3))) * 16;
      dma_glb16(dst, (r.rope[j] >= 0 ? (const unsigned char*)p.kr + (int64_t)r.rope[j] * (DR * 2) : g_few_zero_row) + off);
    }
  };

  // ---- accumulators: O^T, reference and exact max, sum ----
  using AccV = std::conditional_t<HT == 2, f32x16, f32x4>;
  constexpr int NDT = HT == 2 ? D / 32 : D / 16;
  constexpr int NACC = HT == 2 ? 16 : 4;
  AccV acc[NDT];
  float m_ref[HT], m_true[HT], l_run[HT];
#pragma unroll
  for (int ht = 0; ht < HT; ++ht) {
    m_ref[ht] = m_true[ht] = -INFINITY;
    l_run[ht] = 0.f;
  }

  // ---- fragment addresses ----
  const int g1_lane = li * 256 + ((lg ^ nope_swz(li)) * 16);
  const int g1r = NOPE + li * (DR * 2) + ((lg ^ rope_swz(li)) * 16);
  // V^T: each 16-lane group transposes 4 tokens x 16 columns.  32 heads: the
  // group's columns are 16 (g & 1) .. of a 32-column tile, its tokens
  // 8 (g >> 1) .. +3, then +4 .. +7 (16-byte chunk index flips by 3, the
  // swizzle's bit for token bit 2); 16 heads: 16 columns, tokens 4 g .. +3.
  const int tr_row = HT == 2 ? (lg >> 1) * 8 + (li >> 2) : lg * 4 + (li >> 2);
  const int tr_chunk = (HT == 2 ? (lg & 1) * 2 : 0) + ((li & 3) >> 1);
  const int g2_lane = tr_row * 256 + ((tr_chunk ^ nope_swz(tr_row)) * 16) + (li & 1) * 8;
  const int g2b_lane = (tr_row + 4) * 256 + ((tr_chunk ^ nope_swz(tr_row + 4)) * 16) + (li & 1) * 8;
  auto tr_read = [&](const unsigned char* a) -> s16x4 {
    return __builtin_bit_cast(s16x4, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)a));
  };

  // ---- one tile ----
  bool overflow = false, exact_ref = false;
  // GEMM1 of tile t issues the last quarter of tile t + 1 (its buffer was in
  // use until the end of tile t - 1's second product), GEMM2 the rope rows and
  // the first three quarters of tile t + 2, each into a quarter of tile t's
  // buffer whose columns are done.
  auto gemm1 = [&](int b, f32x4 (&s)[HT][2], bool dma1, const Rows& r1) {
    const unsigned char* buf = ring + b * BUFB;
    int g1 = g1_lane;
    asm volatile("" : "+v"(g1));  // the offsets below are not held across tiles
    auto kfrag = [&](int ks) -> V8 {
      if (ks < KSN) return as_v8<V8>(*(const u32x4*)(buf + (g1 ^ ((ks & 3) << 6)) + (ks >> 2) * 4096));
      return as_v8<V8>(*(const u32x4*)(buf + (g1r ^ ((ks - KSN) << 6))));
    };
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) s[ht][0] = s[ht][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // K fragments in flight; with six, the bf16 kernel for 32 heads and four
    // waves copies an accumulator tile between register files in its loop (700
    // rows of 2048 tokens 256 us against 211)
    constexpr int PF = HT == 2 && TW > 1 && kSplitP && BUF ? 4 : 6;
    V8 fa[PF];
#pragma unroll
    for (int i = 0; i < PF; ++i) fa[i] = kfrag(i);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const V8 a = fa[ks % PF];
      if (ks + PF < KS) fa[ks % PF] = kfrag(ks + PF);
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) s[ht][ks & 1] = E::mfma(a, qf[ht][ks], s[ht][ks & 1]);
      if (ks < 4 && dma1) issue_nope(r1, b ^ 1, 3, ks);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // scores of head tile ht in log2 units, lane -> head li, tokens 4 lg + r; returns their max
  auto scaled = [&](const f32x4 (&s)[HT][2], int ht, int nleft, float (&v)[4]) -> float {
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = lg * 4 + r < nleft ? (s[ht][0][r] + s[ht][1][r]) * p.scale_log2 : -INFINITY;
      tmax = fmaxf(tmax, v[r]);
    }
    return xgroup_max(tmax);
  };
  auto run_tile = [&](int b, int nleft, bool with_lo, bool dma1, const Rows& r1, bool dma2, const Rows& r2) {
    const unsigned char* buf = ring + b * BUFB;
    f32x4 s[HT][2];
    gemm1(b, s, dma1, r1);
    int g2 = g2_lane, g2b = g2b_lane;
    asm volatile("" : "+v"(g2), "+v"(g2b));  // the offsets below are not held across tiles
    // the first V^T fragments are on their way during the softmax
    constexpr int PV = 4;
    typedef std::conditional_t<HT == 2, i16x8, s16x4> VFrag;
    auto vfrag = [&](int d) -> VFrag {
      if constexpr (HT == 2) {
        const int o = (d & 3) << 6, c = (d >> 2) * 4096;
        const s16x4 v1 = tr_read(buf + (g2 ^ o) + c), v2 = tr_read(buf + (g2b ^ o) + c);
        return (i16x8){v1[0], v1[1], v1[2], v1[3], v2[0], v2[1], v2[2], v2[3]};
      } else {
        return tr_read(buf + (g2 ^ ((d & 7) << 5)) + (d >> 3) * 4096);
      }
    };
    VFrag va[PV];
#pragma unroll
    for (int i = 0; i < PV; ++i) va[i] = vfrag(i);
    // softmax numerators: lane -> head li (+ 16 ht), tokens 4 lg + r
    T4 hi[HT], lo[HT];
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      float v[4];
      const float tmax = scaled(s, ht, nleft, v);
      m_true[ht] = fmaxf(m_true[ht], tmax);
      if (!exact_ref && m_ref[ht] == -INFINITY) m_ref[ht] = tmax;
      overflow |= tmax > m_ref[ht] + kRefSlack<T>;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = m_ref[ht] == -INFINITY ? 0.f : fast_exp2(v[r] - m_ref[ht]);
        l_run[ht] += e;
        hi[ht][r] = E::from_f32(e);
        lo[ht][r] = E::from_f32(e - E::to_f32(hi[ht][r]));
      }
    }
    // B operand of the second product.  32 heads: rows of 16 lanes hold heads
    // 0-15, 16-31 of tokens 0-7 (lanes 32-63: 8-15) after the swaps
    auto pfrag = [&](const T4 (&pv)[HT]) -> VFrag {
      if constexpr (HT == 2) {
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 x = __builtin_bit_cast(u32x2, pv[0]), y = __builtin_bit_cast(u32x2, pv[HT - 1]);
        const auto w0 = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
        const auto w1 = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
        const u32x4 bw = {w0[0], w1[0], w0[1], w1[1]};
        return __builtin_bit_cast(i16x8, bw);
      } else {
        return __builtin_bit_cast(s16x4, pv[0]);
      }
    };
    auto mfma2 = [&](VFrag v, VFrag b, AccV c) -> AccV {
      if constexpr (HT == 2) return E::mfma32(__builtin_bit_cast(V8, v), __builtin_bit_cast(V8, b), c);
      else return Mfma16<T>::run(v, b, c);
    };
    auto gemm2 = [&](VFrag bp, auto last_pass) {
      constexpr int PQ = NDT / 4;  // d-tiles of a quarter
#pragma unroll
      for (int d = 0; d < NDT; ++d) {
        const VFrag v = va[d % PV];
        if (d + PV < NDT) va[d % PV] = vfrag(d + PV);
        acc[d] = mfma2(v, bp, acc[d]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(last_pass)::value) {
          // the products of quarter q - 1 are issued, so its reads are back
          constexpr int SP = PQ / 4;
          const int q = d / PQ;
          if (dma2) {
            if (q == 0 && d < 2) issue_rope(r2, b, d);
            if (q > 0 && d % SP == 0) issue_nope(r2, b, q - 1, (d % PQ) / SP);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    VFrag bp = pfrag(hi);
    if constexpr (kSplitP)
      if (with_lo) {
        gemm2(bp, std::false_type{});
#pragma unroll
        for (int i = 0; i < PV; ++i) va[i] = vfrag(i);
        bp = pfrag(lo);
      }
    gemm2(bp, std::true_type{});
  };

  // ---- chunks of positions: compact, then run the whole tiles; what is left
  // of a chunk (fewer than TILE tokens) opens the next one's list.
  const int32_t* gtab = p.layout_kv == DSA_LAYOUT_PA_BSND ? p.block_table + (int64_t)ri.b * p.max_blocks : nullptr;
  int n_list = 0, n_total = 0, nt = 0;
  Rows r1 = {};
  // the list of chunk c, its whole tiles nt, and the first two on their way
  // (without the last quarter of the second: r1)
  auto open_chunk = [&](int c, bool last) {
    {
      int phys[RPL];
      unsigned ok = 0;
#pragma unroll
      for (int u = 0; u < RPL; ++u) {
        phys[u] = 0;
        const int pos = c + u * 64 + lane;
        const bool v = ri.active && pos < p1 && sfa_resolve_id(p, ri, ids[u], pos, &phys[u], gtab);
        ok |= (unsigned)v << u;
      }
#pragma unroll
      for (int u = 0; u < RPL; ++u) {
        const bool v = (ok >> u) & 1;
        const unsigned long long m = __ballot(v);
        if (v) list[n_list + __popcll(m & ((1ull << lane) - 1ull))] = phys[u];
        n_list += __popcll(m);
        n_total += __popcll(m);
      }
    }
    // pad to a whole tile; with entries left over from earlier chunks the list
    // can be full to its last entry, and the pad ends there
    if (last && lane < TILE && n_list + lane < LIST) list[n_list + lane] = -1;
    wave_lds_sync();
    if (!last) load_ids(c + kFewChunk);
    nt = last ? (n_list + TILE - 1) / TILE : n_list / TILE;
    if (nt > 0) {
      const Rows r0 = rows_of(0);
#pragma unroll
      for (int j = 0; j < 2; ++j) issue_rope(r0, 0, j);
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) issue_nope(r0, 0, q, j);
    }
    if (nt > 1) {
      r1 = rows_of(1);
#pragma unroll
      for (int j = 0; j < 2; ++j) issue_rope(r1, 1, j);
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) issue_nope(r1, 1, q, j);
    }
  };

  // ---- the reference maxima: the row's first two tiles, scored once for them
  // alone, before the accumulators are in use.  Every wave scores its own, and
  // all take those of the first wave that has any.
  int n_others = 0;  // tokens of the other waves' first chunks
  const bool last0 = p0 + kFewChunk >= p1;
  if (p0 < p1) open_chunk(p0, last0);
  bool primed = nt > 1;  // tile 1 is on its way whole
  if (primed) {
#pragma unroll
    for (int j = 0; j < 4; ++j) issue_nope(r1, 1, 3, j);
  }
#pragma unroll 1
  for (int t = 0; t < min(nt, 2); ++t) {
    if (t == 0 && primed) wait_vmcnt<NDMA>();  // tile 1's
    else wait_vmcnt<0>();
    f32x4 s[HT][2];
    gemm1(t, s, false, r1);
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      float v[4];
      m_ref[ht] = fmaxf(m_ref[ht], scaled(s, ht, n_list - t * TILE, v));
    }
  }
  if constexpr (TW > 1) {
    if (lane == 0) {
      s_cnt[wave] = n_total;
      s_tiles[wave] = nt;
    }
    if (lg == 0) {
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) s_ref[wave][ht * 16 + li] = m_ref[ht];
    }
    lds_barrier();
    int from = 0;
#pragma unroll
    for (int w = TW - 1; w >= 0; --w) {
      n_others += w == wave ? 0 : s_cnt[w];
      from = s_tiles[w] > 0 ? w : from;
    }
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) m_ref[ht] = s_ref[from][ht * 16 + li];
  }

  // Q in VGPRs from here on: left to one register class with the use above,
  // these kernels spilled it (up to 950 bytes of scratch per lane: 17 us more
  // per launch of 130 rows; the others do not, and are 3 % slower with this)
  if constexpr (HT == 2 && (TW > 1 || !BUF)) {
#pragma unroll
    for (int ht = 0; ht < HT; ++ht)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        u32x4 x = as_u4(qf[ht][ks]);
        asm volatile("" : "+v"(x));
        qf[ht][ks] = as_v8<V8>(x);
      }
  }

  // A head whose scores pass the reference max by more than the slack sends
  // the wave through its positions once more, with the exact maxima as
  // references.
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
    for (int d = 0; d < NDT; ++d)
#pragma unroll
      for (int r = 0; r < NACC; ++r) acc[d][r] = 0.f;
    for (int c = p0; c < p1; c += kFewChunk) {
      const bool last = c + kFewChunk >= p1;
      if (pass > 0 || c > p0) open_chunk(c, last);
      // the lo part of P: while the workgroup has seen fewer tokens than the rule says
      const bool with_lo = n_total + n_others < kLoSplitMinTokens || pass > 0;
      Rows r2 = {};
#pragma unroll 1  // (nor peeled for `primed`: a second copy of the loop body spills)
      for (int t = 0; t < nt; ++t) {
        // all of tile t is in; 14 DMAs of tile t + 1 came after it (a later
        // load of the compiler's own only makes this wait longer)
        if (t + 1 < nt) wait_vmcnt<NDMA - 4>();
        else wait_vmcnt<0>();
        if (t + 2 < nt) r2 = rows_of(t + 2);
        run_tile(t & 1, n_list - t * TILE, with_lo, t + 1 < nt && !primed, r1, t + 2 < nt, r2);
        primed = false;
        r1 = r2;
      }
      if (!last) {
        const int done = nt * TILE, left = n_list - done;
        const int keep = lane < left ? list[done + lane] : 0;
        wave_lds_sync();
        if (lane < left) list[lane] = keep;
        n_list = left;
      }
    }
    if (pass > 0 || !__any(overflow)) break;
    exact_ref = true;
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      m_ref[ht] = m_true[ht];
      l_run[ht] = 0.f;
    }
    n_list = n_total = 0;
    load_ids(p0);
  }

  // ---- epilogue ----
#pragma unroll
  for (int ht = 0; ht < HT; ++ht) l_run[ht] = xgroup_sum(l_run[ht]);
  if constexpr (TW == 1) {
    // rows are staged in the ring in the output type and stored whole
    float mul[HT];
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      mul[ht] = l_run[ht] > 0.f ? 1.f / l_run[ht] : 0.f;
      const int head = ht * 16 + li;
      if (p.return_lse && lg == 0 && head < p.n1) {
        const bool any = p.return_lse == 1 && l_run[ht] > 0.f;
        p.smax[row * p.n1 + head] = any ? m_true[ht] * kLn2 : 0.f;
        p.ssum[row * p.n1 + head] = any ? l_run[ht] * fast_exp2(m_ref[ht] - m_true[ht]) : 0.f;
      }
    }
    constexpr int SROW = D * 2 + 16;
    static_assert(HEADS * SROW <= 2 * BUFB, "staging");
    const float mo = HT == 2 ? ((lane & 16) ? mul[HT - 1] : mul[0]) : mul[0];
    const int hrow = HT == 2 ? (lane & 31) : li;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int d = 0; d < NDT; ++d)
#pragma unroll
      for (int q = 0; q < NACC / 4; ++q) {
        const int col = HT == 2 ? d * 32 + q * 8 + (lane >> 5) * 4 : d * 16 + lg * 4;
        const T4 o = {E::from_f32(acc[d][q * 4 + 0] * mo), E::from_f32(acc[d][q * 4 + 1] * mo),
                      E::from_f32(acc[d][q * 4 + 2] * mo), E::from_f32(acc[d][q * 4 + 3] * mo)};
        *(T4*)(ring + hrow * SROW + col * 2) = o;
      }
    wave_lds_sync();
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
      const u32x4 v = *(const u32x4*)(ring + h * SROW + lane * 16);
      if (h < p.n1) *(u32x4*)((unsigned char*)p.out + (row * p.n1 + h) * (D * 2) + lane * 16) = v;
    }
  } else {
    // merge the waves in fp32 through the idle rings: O_w counts 2^(m_ref_w - M)
#pragma unroll
    for (int ht = 0; ht < HT; ++ht)
      if (lg == 0) {
        s_st[wave][0][ht * 16 + li] = m_ref[ht];
        s_st[wave][1][ht * 16 + li] = l_run[ht];
        s_st[wave][2][ht * 16 + li] = m_true[ht];
      }
    __syncthreads();
    auto weight = [&](int w, int h, float M) -> float {  // a wave without tokens counts nothing
      return s_st[w][1][h] == 0.f ? 0.f : fast_exp2(s_st[w][0][h] - M);
    };
    auto top = [&](int h) {
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < TW; ++w) M = s_st[w][1][h] == 0.f ? M : fmaxf(M, s_st[w][0][h]);
      return M;
    };
    const int hown = HT == 2 ? (lane & 31) : li;
    const float fw = weight(wave, hown, top(hown));
    // all columns of 16 heads (half the columns of 32) fit the rings at once;
    // wave w then sums heads w HPW .. of all waves, 4 columns per lane at a time
    constexpr int CB = D / HT, NR = HT;
    constexpr int FROW = CB + 4;                     // floats of a staged head row
    constexpr int HPW = HEADS / TW;
    constexpr int UPR = 2 / NR;                      // 256-column pieces per round
    static_assert(TW * HEADS * FROW * 4 <= TW * 2 * BUFB, "staging");
    float* const stg = (float*)&smem[0][0];
    f32x4 res[HPW][2];
#pragma unroll
    for (int rd = 0; rd < NR; ++rd) {
      if (rd > 0) __syncthreads();
      constexpr int DPR = NDT / NR;
#pragma unroll
      for (int dd = 0; dd < DPR; ++dd)
#pragma unroll
        for (int q = 0; q < NACC / 4; ++q) {
          const int d = rd * DPR + dd;
          const int col = HT == 2 ? dd * 32 + q * 8 + (lane >> 5) * 4 : dd * 16 + lg * 4;
          f32x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = acc[d][q * 4 + r] * fw;
          *(f32x4*)(stg + (wave * HEADS + hown) * FROW + col) = o;
        }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < HPW; ++i)
#pragma unroll
        for (int u = 0; u < UPR; ++u) {
          const int h = wave * HPW + i;
          f32x4 a = *(const f32x4*)(stg + h * FROW + u * 256 + lane * 4);
#pragma unroll
          for (int w = 1; w < TW; ++w) a += *(const f32x4*)(stg + (w * HEADS + h) * FROW + u * 256 + lane * 4);
          res[i][rd + u] = a;
        }
    }
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
      const int h = wave * HPW + i;
      if (h >= p.n1) break;
      const float M = top(h);
      float L = 0.f, mt = -INFINITY;
#pragma unroll
      for (int w = 0; w < TW; ++w) {
        L += s_st[w][1][h] * weight(w, h, M);
        mt = fmaxf(mt, s_st[w][2][h]);
      }
      const float inv = L > 0.f ? 1.f / L : 0.f;
      const int64_t orow = row * p.n1 + h;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const f32x4 v = res[i][u] * inv;
        const T4 o = {E::from_f32(v[0]), E::from_f32(v[1]), E::from_f32(v[2]), E::from_f32(v[3])};
        *(T4*)((T*)p.out + orow * D + u * 256 + lane * 4) = o;
      }
      if (lane == 0 && p.return_lse) {
        const bool any = p.return_lse == 1 && L > 0.f;
        p.smax[orow] = any ? mt * kLn2 : 0.f;
        p.ssum[orow] = any ? L * fast_exp2(M - mt) : 0.f;
      }
    }
  }
}

template <typename T, int HT, int TW>
void launch_one(const SfaFwdParams& p, bool buf, unsigned blocks, hipStream_t stream) {
  if (buf) hipLaunchKernelGGL((sfa_fwd_few_kernel<T, HT, TW, true>), dim3(blocks), dim3(TW * 64), 0, stream, p);
  else hipLaunchKernelGGL((sfa_fwd_few_kernel<T, HT, TW, false>), dim3(blocks), dim3(TW * 64), 0, stream, p);
}

}  // namespace

int sfa_few_heads_per_wg(int64_t n1) { return n1 <= 16 ? 16 : 32; }

hipError_t sfa_few_launch(const SfaFwdParams& p, int32_t dtype, bool buf, int64_t rows_per_xcd, hipStream_t stream) {
  const int hpw = sfa_few_heads_per_wg(p.n1);
  const unsigned blocks = (unsigned)(8 * rows_per_xcd);
  // One wave per row once the rows come near filling every SIMD (16 heads,
  // 2048 tokens: 179 against 229 us at 800 rows); below that a workgroup's
  // four waves share a row's tokens (600 rows: 173 against 176 us; 1024 tokens,
  // 500 rows 74 against 92).  With short rows, whose start and merge weigh more,
  // the line lies lower (700 causal rows of up to 512 tokens: one wave 50 us,
  // four 65; 1024 tokens: 95 and 108).
  const int64_t per_cu = (int64_t)p.K * p.bs <= 1024 ? 2 : 3;
  const bool one = p.rows > per_cu * device_cu_count();
  auto go = [&](auto t) {
    using T = decltype(t);
    if (hpw == 16) one ? launch_one<T, 1, 1>(p, buf, blocks, stream) : launch_one<T, 1, 4>(p, buf, blocks, stream);
    else one ? launch_one<T, 2, 1>(p, buf, blocks, stream) : launch_one<T, 2, 4>(p, buf, blocks, stream);
  };
  if (dtype == DSA_DTYPE_BF16) go(bf16{});
  else go(f16{});
  return hipGetLastError();
}

}  // namespace dsa
