// Parameters, row order and DMA helpers shared by the sparse flash attention
// forward kernels (sfa_fwd.hip: 64 / 128 heads per workgroup; sfa_fwd_few.hip:
// up to 32).
#pragma once

#include "common.h"
#include "sfa_common.h"

namespace dsa {

struct SfaFwdParams {
  const void* q;
  const void* qr;
  const void* k;
  const void* kr;
  const int32_t* idx;
  const int32_t* act_q;
  const int32_t* act_k;
  const int32_t* block_table;
  void* out;
  float* smax;
  float* ssum;
  // split partials (splits > 1): part_o[s, r, h, :] = O_s / (l_s * scale_s)
  // in fp16, scale_s = 2^e >= max |O_s / l_s| (so |values| < 1: fp16 keeps
  // 11 bits for the largest ones); part_ml[s, r, h] = {reference max (log2
  // units), l_s, exact max (log2 units), scale_s}
  _Float16* part_o;
  float* part_ml;
  int64_t rows;
  int64_t kv_rows;
  int32_t batch, s1, s2, n1, K;
  int32_t bs;  // sparse_block_size
  int32_t mode, layout_q, layout_kv;
  int64_t band_pre, band_next;  // pre_tokens / next_tokens clamped to +-kBandOpen
  int32_t max_blocks, page_size;
  int32_t splits, pos_per_split;
  int32_t lo_range;   // > 0: the lo part's rule holds for ranges of this length (SfaLoProbe)
  int32_t row_shift;  // 2^row_shift consecutive rows go to one XCD in turn (sfa_block_row)
  float scale_log2;
  int32_t return_lse;  // 0: no statistics, 1: the statistics, 2: zeros
};

// Row of slot j of an XCD (workgroup x runs on XCD x % 8): blocks of
// 2^row_shift consecutive rows go to the XCDs in turn, the last rows first.
// Under a causal mask the first rows of a sequence are short: given one
// contiguous range of rows each, XCD 0 ran out of work at a quarter of the
// others' (by token counts 0.75 of the chip's time used at 4096 rows of up to
// 2048 tokens, 0.875 at 8192), and rows in ascending order left the longest
// ones for the last round: 8192 rows of 128 heads 4.34 -> 4.02 ms.  Blocks keep the rows that run together on an XCD adjacent
// (neighbouring rows select much the same keys, which its L2 then holds).
__device__ __forceinline__ int64_t sfa_block_row(const SfaFwdParams& p, int xcd, int j) {
  const int sh = p.row_shift;
  const int64_t i = (((int64_t)(j >> sh) * 8 + xcd) << sh) + (j & ((1 << sh) - 1));
  return p.rows - 1 - i;
}

// P carries a bf16 lo part (the P.V product then has ~16 bits of P) only
// while a workgroup attends fewer tokens than this; from here on P is
// rounded once to bf16, as the reference kernel rounds it
// (sparse_flash_attention_triton.py:313-323).  The rounding error of O is
// then ~2^-9 |v| / sqrt(3 n_eff) with n_eff the effective number of tokens
// of the softmax, far below the fp32-golden tolerance (atol 2e-3) at these
// lengths, while for a handful of tokens it is not.
constexpr int kLoSplitMinTokens = 256;

// The same rule where a launch takes fewer, longer ranges than the split count
// rounded up: P keeps its lo part wherever it would have it in that count's
// ranges (of lo_range positions).  A workgroup drops it only if every position
// of its own range is attended, and so are enough beyond both ends to fill the
// first and the last of those ranges that it touches up to the limit: one
// probed position per thread, loaded beside the workgroup's own (0.5 us per
// launch; counting every touched range took 2, and the lo part in all
// workgroups 4 of 29).
template <int NTHR>
struct SfaLoProbe {
  static constexpr int kN = 2 * kLoSplitMinTokens / NTHR;
  int pos[kN], id[kN];  // pos < 0: nothing to probe
  template <typename P>
  __device__ __forceinline__ void load(const P& p, const int32_t* idx_row, int p0, int p1, int tid) {
    const int total = p.K * p.bs, r = p.lo_range;
    const int end = (p1 - 1) / r * r + kLoSplitMinTokens;         // the last range's limit
    const int beg = min(p1, p0 / r * r + r) - kLoSplitMinTokens;  // the first range's, from its end
#pragma unroll
    for (int u = 0; u < kN; ++u) {
      const int i = u * NTHR + tid;
      const int x = i < kLoSplitMinTokens ? p1 + i : p0 + kLoSplitMinTokens - 1 - i;
      pos[u] = (i < kLoSplitMinTokens ? x < end : x >= max(beg, 0)) ? x : -1;
      id[u] = pos[u] >= 0 && x < total ? sfa_load_id(p, idx_row, x) : -1;
    }
  }
  // whether a position that this wave probed is not attended
  template <typename P>
  __device__ __forceinline__ bool missing(const P& p, const RowInfo& ri) const {
    bool miss = false;
#pragma unroll
    for (int u = 0; u < kN; ++u) {
      int64_t tok;
      miss |= pos[u] >= 0 && !(ri.active && sfa_visible(p, ri, id[u], pos[u], &tok));
    }
    return __any(miss);
  }
};
// How far (log2 units) a score may pass a head's reference max: the numerators
// 2^(s - m_ref) go to the second product in T, whose largest power of two is
// 2^127 (bf16; the fp32 sums keep the rest of the range) or 2^15 (fp16).
template <typename T> constexpr float kRefSlack = 64.f;
template <> inline constexpr float kRefSlack<f16> = 15.f;
// Smallest exponent of a split partial's scale 2^e: a partial whose largest
// |O / l| is below 2^kPartMinExp (tiny values) keeps the scale 2^-120, so
// the stored multiplier inv * 2^-e (inv <= 1: l counts the reference-max
// token) stays finite and the stored values stay below 1.
constexpr int kPartMinExp = -120;

// One 16-byte-per-lane DMA from global memory straight into LDS: lane L's
// 16 bytes land at lds_base + 16*L (LDS address taken from M0).  Issued via
// inline asm so that the compiler does not drain all outstanding DMA before
// every LDS read; the tile loop waits with explicit vmcnt counts instead.
__device__ __forceinline__ void dma_buf16(unsigned lds_base, int voff, __amdgpu_buffer_rsrc_t rsrc) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds_base), "v"(voff), "s"(rsrc) : "memory");
}
__device__ __forceinline__ void dma_glb16(unsigned lds_base, const void* gaddr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(lds_base), "v"(gaddr) : "memory");
}
template <int N> __device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

// sfa_fwd_few.hip: D = 512 kernels for few heads (no token splits)
int sfa_few_heads_per_wg(int64_t n1);
hipError_t sfa_few_launch(const SfaFwdParams& p, int32_t dtype, bool buf, int64_t rows_per_xcd, hipStream_t stream);

}  // namespace dsa
