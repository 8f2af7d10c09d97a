// Segmented attention for fp32 q and k at the default dot modes (16-bit V, or
// fp32 V split like K): split-bf16 products fed by DMA, software-pipelined.
//
// K arrives as split rows (dtype code kSplitRows): each row of 128 fp32
// values is stored as its 128 bf16 high parts, then its 128 bf16 low parts
// (hi = x rounded to bf16, lo = (x - hi) rounded to bf16; 512 bytes, the size
// of the fp32 row).  split_rows_kernel writes them from fp32 rows; q is split
// the same way when it is loaded.  S = Kh Qh + Kh Ql + Kl Qh then carries
// about 16 significand bits, as the register-staged kernel's 2-piece split
// (seg_attn_staged.hip) does, without re-splitting every K tile for every
// query tile.
//
// Layout and schedule (CDNA4, wave64), one workgroup of 8 waves x 32 queries
// (256 queries of one (b, h)) per CU:
//  * A 64-key tile moves global -> LDS with buffer_load_dwordx4 ... lds in
//    MFMA-operand order: the hi plane and the lo plane of K (16 KiB each, the
//    16-bit kernel's K block order) and V (16 KiB, the 16-bit kernel's V
//    order, read with ds_read_b64_tr_b16).  K has two stages, V three slots:
//    112 KiB.
//  * The software pipeline runs on 32-key halves: half j+1's 24 QK MFMAs
//    (8 k-steps x 3 products) are issued while the VALU turns half j's
//    scores into P, then half j's 8 PV MFMAs while the VALU takes half j+1's
//    row max.  Two S halves of 16 registers each, so both q pieces (64
//    registers) and O (64) fit 256 registers per wave.
//  * K of tile T is read by the half steps 2T - 1 and 2T, V of tile T by 2T
//    and 2T + 1.  Step 2T + 1 waits for tile T + 1 (issued two half steps
//    earlier), passes the tile's one barrier, which retires every read of
//    K(T) and V(T - 1), and issues K and V of tile T + 2 into their places:
//    each tile lands at least two half steps before its first use, and the
//    even half steps neither wait nor synchronize.
// Semantics as the other attention kernels (attn_common.h): online softmax in
// the exp2 domain with the lazy rescale, P rounded to V's type, current-scale
// tiles first, then the retained prior rows through the row tables.
#include "attn_common.h"

#include <type_traits>

namespace hkv {
namespace {

using namespace attn;

constexpr int kSW = 8;                           // waves per workgroup
constexpr int kSThreads = kSW * 64;
constexpr int kSBM = kSW * 32;                   // queries per item
constexpr int kSPlane = kBN * kD * 2;            // 16 KiB: one plane of a K tile
constexpr int kSKStage = 2 * kSPlane;            // K hi and lo planes of a tile
constexpr int kSVBase = 2 * kSKStage;            // V slots after the two K stages
constexpr int kSRing = kSVBase + 3 * kSPlane;    // 2 K stages + 3 V slots: 112 KiB
constexpr int kSRowBytes = 2 * kD * 2;           // a split K row
constexpr int kVRowBytes = kD * 2;               // a 16-bit V row
constexpr int32_t kPastEnd = static_cast<int32_t>(0x80000000u);

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4_ptr;
typedef __attribute__((address_space(3))) void* lds_void_ptr;

__device__ __forceinline__ u32x2_t ds_read_tr(const uint8_t* p) {
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p)));
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_ptr)(p)));
}

// 16 bytes per lane from a buffer straight to LDS at `lds_addr` + 16 lane
// (see seg_attn_direct.hip: inline assembly so that LDS reads are not made
// to wait for every outstanding load; M0 is used by nothing else here).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const u32x4_t rsrc, uint32_t lds_addr, int32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(rsrc)
               : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ u32x4_t make_desc(const void* base, uint32_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  u32x4_t d;
  d[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p));
  d[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p >> 32) & 0xffffu);
  d[2] = __builtin_amdgcn_readfirstlane(bytes);
  d[3] = 0x00020000u;
  return d;
}

// Keys of half kb (32kb .. 32kb + 31) at or past `valid_keys` (of the tile) get -inf.
__device__ __forceinline__ void mask_half(f32x16_t& s, int kb, int valid_keys, int g) {
  const int lim = valid_keys - 32 * kb - 4 * g;
#pragma unroll
  for (int j = 0; j < 16; ++j)
    if (8 * (j >> 2) + (j & 3) >= lim) s[j] = -__builtin_inff();
}

__device__ __forceinline__ float half_max(const f32x16_t& s) {
  float mx = s[0];
#pragma unroll
  for (int j = 1; j < 16; ++j) mx = fmaxf(mx, s[j]);
  return pair_max(mx);
}

// p = exp2(c (s - m)) in place, l_run += sum of p (fp32, unrounded).
__device__ __forceinline__ void exp_half(f32x16_t& s, float m_run, float c, float& l_run) {
  const float mc = m_run * c;
#pragma unroll
  for (int j = 0; j < 16; ++j) s[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j], c, -mc));
  float p0 = s[0], p1 = s[8];
#pragma unroll
  for (int j = 1; j < 8; ++j) {
    p0 += s[j];
    p1 += s[8 + j];
  }
  l_run += p0 + p1;
}

// fp32 row -> split row: 16 threads per row, 8 values each (thread c of the row).
__device__ __forceinline__ void split_row(const float* src, uint8_t* dst, int64_t row, int c) {
  const f32x4_t x = *reinterpret_cast<const f32x4_t*>(src + row * kD + c * 8);
  const f32x4_t y = *reinterpret_cast<const f32x4_t*>(src + row * kD + c * 8 + 4);
  const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  u32x4_t hi, lo;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    hi[k] = pack2<kBF16>(v[2 * k], v[2 * k + 1]);
    const float h0 = __builtin_bit_cast(float, hi[k] << 16);
    const float h1 = __builtin_bit_cast(float, hi[k] & 0xffff0000u);
    lo[k] = pack2<kBF16>(v[2 * k] - h0, v[2 * k + 1] - h1);
  }
  uint8_t* const out = dst + row * kSRowBytes;
  *reinterpret_cast<u32x4_t*>(out + c * 16) = hi;
  *reinterpret_cast<u32x4_t*>(out + kD * 2 + c * 16) = lo;
}

__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ src, uint8_t* __restrict__ dst,
                                                         int64_t rows) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >> 4 < rows) split_row(src, dst, i >> 4, static_cast<int>(i & 15));
}

// What an attention call on fp32 K (and V) rows splits before it: the current
// rows, and of the slab only the rows that the tables' segments hold, K and V
// (blockIdx.y) in one launch.  HBM bound.  A block of current rows moves 16, one
// per 16 threads: short blocks, many in flight.  A block of the slab owns 32
// consecutive rows of it: its threads mark in one word of LDS which of them any
// head's segment holds (one round trip for the tables, all entries at once) and
// move those; every block does about the same, however the rows are spread over
// the heads.  The slab's blocks come first, as they wait for the tables.  Whole
// calls, B=2, 16 heads: 2272 tokens, fp32 q/k, heads of very different retained
// lengths 224.8 -> 215.5 us against each head's rows walked as one stream by 16
// blocks of 64-row steps (216.5 with every slab row split, in two launches);
// 2304 tokens all fp32, a tenth retained 323 -> 318 us.  Non-temporal stores
// cost 1 to 3 % of a call: the attention reads the rows next.
constexpr int kSplitCurRows = 16;
constexpr int kSplitSlabRows = 32;

__global__ __launch_bounds__(256) void split_operands_kernel(const SplitOperands o) {
  __shared__ uint32_t live;
  const bool is_v = blockIdx.y != 0;
  const int tid = threadIdx.x;
  const int sub = tid >> 4, c = tid & 15;
  const int64_t blk = blockIdx.x;
  if (blk >= o.slab_blocks) {
    const int64_t row = (blk - o.slab_blocks) * kSplitCurRows + sub;
    if (row < o.cur_rows) split_row(is_v ? o.cur_v : o.cur_k, is_v ? o.cur_v_out : o.cur_k_out, row, c);
    return;
  }
  const int64_t cap = o.slab_capacity;
  const int64_t b = blk / o.slab_chunks;
  const int64_t r0 = (blk - b * o.slab_chunks) * kSplitSlabRows;
  if (tid == 0) live = 0;
  __syncthreads();
  uint32_t mine = 0;
  for (int32_t e = tid; e < o.heads * o.max_segments; e += 256) {
    const int32_t h = e / o.max_segments;
    // rows [st, en) of the entry, clamped to the slab as the attention clamps them
    int64_t st = o.seg_starts[e], en = o.seg_ends[e];
    if (e - h * o.max_segments >= o.seg_counts[h]) continue;
    st = (st < 0 ? 0 : st) - r0;
    en = (en > cap ? cap : en) - r0;
    st = st < 0 ? 0 : st;
    en = en > kSplitSlabRows ? kSplitSlabRows : en;
    if (en > st) mine |= static_cast<uint32_t>(((1ull << (en - st)) - 1) << st);
  }
  if (mine != 0) atomicOr(&live, mine);
  __syncthreads();
  const uint32_t rows = live;
  const float* const src = is_v ? o.slab_v : o.slab_k;
  uint8_t* const dst = is_v ? o.slab_v_out : o.slab_k_out;
#pragma unroll
  for (int u = 0; u < kSplitSlabRows / 16; ++u)
    if ((rows >> (sub + 16 * u)) & 1) split_row(src, dst, b * cap + r0 + sub + 16 * u, c);
}

template <int VDT>
__global__ __launch_bounds__(kSThreads, 1) void seg_attn_split_kernel(const int32_t* __restrict__ plan_p,
                                                                     const int32_t n_units, const AttnArgs a,
                                                                     const Scalars sc,
                                                                     const int32_t n_qt) {
  constexpr int kThreads = kSThreads;
  constexpr int kBM = kSBM;
  constexpr int MV = VDT;
  __shared__ __attribute__((aligned(1024))) uint8_t ring[kSRing];
  __shared__ __attribute__((aligned(16))) int32_t rowtab[3][kBN];
  __shared__ int32_t seg_start[kMaxSegments];
  __shared__ int32_t seg_pref[kMaxSegments + 1];
  __shared__ int32_t merge_turn;
  static_assert(kSRing >= kSW * 32 * kOutPitch, "output staging fits the ring");

  const int64_t cap = a.slab_capacity;
  const int H = a.heads;
  const int L = a.cur_len;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform by construction
  const int g = lane >> 5;
  // This workgroup's plan unit, loaded with the kernel arguments: the plan
  // pointer and unit count are preloaded into SGPRs (as in the 16-bit
  // kernel).
  int32_t pu[kPlanInts] = {};
  const bool planned = plan_p != nullptr && static_cast<int32_t>(blockIdx.x) < n_units;
  if (planned) {
    const int32_t* src = plan_p + static_cast<int64_t>(blockIdx.x) * kPlanInts;
#pragma unroll
    for (int i = 0; i < kPlanInts; ++i) pu[i] = src[i];
  }

  // The unit: from the caller's work plan (a whole item or one key-range
  // part of a cut item, merged through the workspace), else the workgroup's
  // item in longest-first order.
  WorkItem w;
  Unit un{0, 0, 1, 0, 0, 0};
  int32_t p0 = 0, p1 = 0;
  if (planned) {
    const int32_t ph = pu[0], pj = pu[1], pcut = pu[4], ppart = pu[5];
    p0 = pu[2];
    p1 = pu[3];
    if (ph < 0 || ph >= H || pj < 0 || pj >= a.batch * n_qt) return;  // not a unit of this launch
    w.h = ph;
    w.b = pj / n_qt;
    w.qt = pj - w.b * n_qt;
    w.bh = w.b * H + w.h;
    const bool cut = pcut >= 0 && a.workspace != nullptr && pcut < a.ws_cuts && ppart >= 0 && ppart < 2;
    un.part = cut ? ppart : 0;
    un.parts = cut ? 2 : 1;
    un.record = cut ? 2 * pcut : 0;
    un.counter = cut ? pcut : 0;
    un.arrive = cut && pu[7] != 0 ? 1 : 0;
    load_head_segments<kThreads>(a.seg_starts, a.seg_ends, a.seg_counts, cap, a.max_segments, w, seg_start,
                                 seg_pref);
  } else {
    int32_t* head_rows = reinterpret_cast<int32_t*>(ring);
    w = plan_work<kThreads>(a.seg_starts, a.seg_ends, a.seg_counts, cap, H, a.max_segments, a.batch, n_qt,
                            head_rows, head_rows + kMaxHeads, seg_start, seg_pref,
                            static_cast<int32_t>(blockIdx.x), head_rows + 2 * kMaxHeads,
                            kSRing / 4 - 2 * kMaxHeads);
  }
  const int32_t R = w.R;
  const int32_t ntc = (L + kBN - 1) / kBN;
  const int32_t ntiles = (R + kBN - 1) / kBN + ntc;
  const int32_t parts = un.parts;
  int32_t tb = 0, te = ntiles;
  if (parts > 1) {
    tb = p0 < 0 ? 0 : (p0 > ntiles ? ntiles : p0);
    te = p1 < tb ? tb : (p1 > ntiles ? ntiles : p1);
  }
  const int32_t qrow = w.qt * kBM + wave * 32 + (lane & 31);
  if (tb >= te) {
    // a planned part with no key tiles (a plan that does not match these
    // tables): its record is empty -- zero weight in the merge
    f32x16_t none[4] = {};
    merge_parts<kF32, kThreads>(a, sc, un, parts, none, -1e30f, 0.f, w, qrow, L, H, g, merge_turn,
                                ring + wave * 32 * kOutPitch);
    return;
  }

  // Descriptors: K split rows and V rows of the slab (batch row b) and of
  // the current scale (b, h).
  const int64_t cur_row0 = static_cast<int64_t>(w.bh) * L;
  const u32x4_t dk_prior = make_desc(static_cast<const uint8_t*>(a.slab_k) + w.b * cap * kSRowBytes,
                                     static_cast<uint32_t>(cap * kSRowBytes));
  const u32x4_t dv_prior = make_desc(static_cast<const uint8_t*>(a.slab_v) + w.b * cap * kVRowBytes,
                                     static_cast<uint32_t>(cap * kVRowBytes));
  const uint8_t* const k_cur = static_cast<const uint8_t*>(a.cur_k) + cur_row0 * kSRowBytes;
  const uint8_t* const v_cur = static_cast<const uint8_t*>(a.cur_v) + cur_row0 * kVRowBytes;

  // This wave's DMA share of a tile: K blocks 4 wave .. + 3 (blocks 0..15 of
  // the hi plane, 16..31 of the lo plane) and V chunks 2 wave, 2 wave + 1.
  int k_key[4], k_col[4], v_key[2], v_col[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = 4 * wave + i;
    const int blk = q & 15;
    k_key[i] = (blk >> 3) * 32 + (lane & 31);
    k_col[i] = (q >> 4) * (kD * 2) + (blk & 7) * 32 + (lane >> 5) * 16;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int qv = 2 * wave + i;
    const int lp = lane & 31;
    const int db = 2 * (qv & 1) + (lane >> 5);
    v_key[i] = 16 * (qv >> 2) + 8 * ((qv >> 1) & 1) + 4 * (lp >> 4) + ((lp & 7) >> 1);
    v_col[i] = 2 * (db * 32 + 16 * ((lp >> 3) & 1) + 8 * (lp & 1));
  }
  const uint32_t ring_lds = lds_address(ring);

  auto issue_k = [&](int T) {
    const uint32_t dst = ring_lds + (T & 1) * kSKStage + wave * 4 * 1024;
    if (T < ntc) {
      const uint32_t skip = static_cast<uint32_t>(T) * (kBN * kSRowBytes);
      const u32x4_t d = make_desc(k_cur + skip, static_cast<uint32_t>(L) * kSRowBytes - skip);
#pragma unroll
      for (int i = 0; i < 4; ++i) dma16(d, dst + i * 1024, k_key[i] * kSRowBytes + k_col[i]);
    } else {
      const int32_t* rt = rowtab[(T - ntc) % 3];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int32_t row = rt[k_key[i]];
        dma16(dk_prior, dst + i * 1024, row < 0 ? kPastEnd : row * kSRowBytes + k_col[i]);
      }
    }
  };
  auto issue_v = [&](int T) {
    const uint32_t dst = ring_lds + kSVBase + (T % 3) * kSPlane + wave * 2 * 1024;
    if (T < ntc) {
      const uint32_t skip = static_cast<uint32_t>(T) * (kBN * kVRowBytes);
      const u32x4_t d = make_desc(v_cur + skip, static_cast<uint32_t>(L) * kVRowBytes - skip);
#pragma unroll
      for (int i = 0; i < 2; ++i) dma16(d, dst + i * 1024, v_key[i] * kVRowBytes + v_col[i]);
    } else {
      const int32_t* rt = rowtab[(T - ntc) % 3];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int32_t row = rt[v_key[i]];
        dma16(dv_prior, dst + i * 1024, row < 0 ? kPastEnd : row * kVRowBytes + v_col[i]);
      }
    }
  };
  auto valid_of = [&](int T) { return T < ntc ? min(kBN, L - T * kBN) : min(kBN, R - (T - ntc) * kBN); };
  int cur_seg = 0;
  auto fill = [&](int T) {  // wave 0: row table of tile T (a prior-row tile)
    if (T >= ntc && T < te)
      fill_rowtab<1>(T - ntc, rowtab[(T - ntc) % 3], cur_seg, w.nseg, R, seg_start, seg_pref, -1);
  };

  // Q in two bf16 pieces: B operands of S^T = K Q^T (query row, d = 16ks + 8g .. +7)
  u32x4_t qh[8], ql[8];
  {
    const __amdgpu_buffer_rsrc_t rq = make_rsrc(static_cast<const uint8_t*>(a.q) + cur_row0 * kD * 4,
                                                static_cast<uint32_t>(L * kD * 4));
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      load8_split(rq, qrow < L ? (qrow * kD + ks * 16 + g * 8) * 4 : -1, qh[ks], ql[ks]);
  }
  if (wave == 0) {
    fill(tb);
    fill(tb + 1);
  }
  __syncthreads();
  issue_k(tb);
  issue_v(tb);
  if (tb + 1 < te) {
    issue_k(tb + 1);
    issue_v(tb + 1);
  }
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    qh[ks] ^= sc.q_sign;
    ql[ks] ^= sc.q_sign;
  }

  f32x16_t oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) oacc[i] = f32x16_t{};
  float m_run = -1e30f;
  float l_run = 0.f;

  // S^T of half j (keys 32 (j & 1) .. of tile j >> 1) from its stage
  auto qk = [&](f32x16_t& s, int j) {
    const uint8_t* kst = ring + ((j >> 1) & 1) * kSKStage + (j & 1) * 8 * 1024 + lane * 16;
    s = f32x16_t{};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const u32x4_t kh = *reinterpret_cast<const u32x4_t*>(kst + ks * 1024);
      const u32x4_t kl = *reinterpret_cast<const u32x4_t*>(kst + kSPlane + ks * 1024);
      s = mfma32<kBF16>(kh, qh[ks], s);
      s = mfma32<kBF16>(kh, ql[ks], s);
      s = mfma32<kBF16>(kl, qh[ks], s);
    }
  };
  // O^T += V^T P^T over half j's keys (k-steps u = 2 (j & 1), + 1)
  auto pv = [&](const f32x16_t& s, int j) {
    const uint8_t* vst = ring + kSVBase + ((j >> 1) % 3) * kSPlane + lane * 8;
#pragma unroll
    for (int ul = 0; ul < 2; ++ul) {
      u32x4_t pf;
      pf[0] = pack2<MV>(s[8 * ul + 0], s[8 * ul + 1]);
      pf[1] = pack2<MV>(s[8 * ul + 2], s[8 * ul + 3]);
      pf[2] = pack2<MV>(s[8 * ul + 4], s[8 * ul + 5]);
      pf[3] = pack2<MV>(s[8 * ul + 6], s[8 * ul + 7]);
      const int u = 2 * (j & 1) + ul;
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const int blk = (db >> 1) * 1024 + (db & 1) * 512;
        const u32x2_t lo = ds_read_tr(vst + (u * 4 + 0) * 1024 + blk);
        const u32x2_t hi = ds_read_tr(vst + (u * 4 + 2) * 1024 + blk);
        const u32x4_t vf = {lo[0], lo[1], hi[0], hi[1]};
        oacc[db] = mfma32<MV>(vf, pf, oacc[db]);
      }
    }
  };
  auto masked_max = [&](f32x16_t& s, int j) {
    float mx = half_max(s);
    asm volatile("" : "+v"(mx));
    const int v = valid_of(j >> 1);
    if (v < 32 * ((j & 1) + 1)) {
      mask_half(s, j & 1, v, g);
      mx = half_max(s);
    }
    return mx;
  };

  // Prologue: tile tb landed (tile tb + 1 may be in flight: 6 DMAs per wave); S of half 2 tb and its max.
  if (tb + 1 < te) wait_vmcnt<6>();
  else wait_vmcnt<0>();
  __syncthreads();
  f32x16_t sa, sb;
  qk(sa, 2 * tb);
  move_max(oacc, m_run, l_run, masked_max(sa, 2 * tb), sc.c, sc.thresh);

  const int jend = 2 * te;
  // Half step j: scur = S(j) (max applied), snext receives S(j + 1) unless j
  // is the item's last half (kMore false: peeled, so that the steps of the
  // loop have no branch between their MFMAs and their softmax).
  auto step = [&](auto more_tag, f32x16_t& scur, f32x16_t& snext, int j) {
    constexpr bool kMore = decltype(more_tag)::value;
    const int T = j >> 1;
    // Waves w and w + 4 share a SIMD, whose issue favours the older wave:
    // left alone, waves 0-3 finish each tile ~1.1 us ahead and wait at its
    // barrier while waves 4-7 run one to a SIMD.  Raising waves 0-3 in the
    // even half steps and waves 4-7 in the odd ones (which start at the
    // barrier) keeps the pairs within ~0.3 us (-1.8 % on the 2B final step
    // at the model's precision).
    if (((j + (wave >> 2)) & 1) == 0)
      __builtin_amdgcn_s_setprio(1);
    else
      __builtin_amdgcn_s_setprio(0);
    if ((j & 1) == 0) {
      // tile T landed at step 2T - 1 (or in the prologue): no wait here
      if (wave == 0) fill(T + 2);
    } else {
      // tile T + 1 (the next half's K, the next step's V), issued two half
      // steps ago, is the only one in flight; after the barrier every read
      // of K(T) and V(T - 1) is done, so tile T + 2 takes their places
      wait_vmcnt<0>();
      __syncthreads();
      if (T + 2 < te) {
        issue_k(T + 2);
        issue_v(T + 2);
      }
    }
    if constexpr (kMore) qk(snext, j + 1);
    exp_half(scur, m_run, sc.c, l_run);
    pv(scur, j);
    if constexpr (kMore) {
      asm volatile("" : "+v"(l_run));
      move_max(oacc, m_run, l_run, masked_max(snext, j + 1), sc.c, sc.thresh);
    }
  };
  using More = std::integral_constant<bool, true>;
  using Last = std::integral_constant<bool, false>;
  int j = 2 * tb;
  for (; j + 2 < jend; j += 2) {
    step(More{}, sa, sb, j);
    step(More{}, sb, sa, j + 1);
  }
  step(More{}, sa, sb, j);
  step(Last{}, sb, sa, j + 1);
  __builtin_amdgcn_s_setprio(0);

  if (parts == 1) {
    if (a.out_dtype != kF32 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0) {
      __syncthreads();  // every wave is past its last tile: the ring is free
      uint8_t* const stage = ring + wave * 32 * kOutPitch;
      const int32_t qrow0 = w.qt * kBM + wave * 32;
      if (a.out_dtype == kF16)
        write_output_lds<kF16>(oacc, m_run, l_run, sc.c, a.out, a.lse, w.b, w.h, qrow0, L, H, w.bh, lane, stage);
      else
        write_output_lds<kBF16>(oacc, m_run, l_run, sc.c, a.out, a.lse, w.b, w.h, qrow0, L, H, w.bh, lane, stage);
    } else {
      write_output(oacc, m_run, l_run, sc.c, a.out, a.lse, w.b, w.h, qrow, L, H, w.bh, g, a.out_dtype);
    }
    return;
  }
  merge_parts<kF32, kThreads>(a, sc, un, parts, oacc, m_run, l_run, w, qrow, L, H, g, merge_turn,
                              ring + wave * 32 * kOutPitch);
}

// ---------------------------------------------------------------- 128-query form
//
// The same products and softmax for items of 128 queries: 4 waves x 32
// queries, two workgroups per CU, and the key stream in 32-key halves (half
// j = keys 32 (j & 1) .. of tile j >> 1), so that fp32 V fits too: with VDT
// kSplitRows V arrives as split rows like K, P is split the same way and
// O += Vh Ph + Vl Ph + Vh Pl (the staged kernel's 2-piece products of fp32 V).
// Bound by the MFMAs: fp32 V takes 48 of them per half (24 QK, 24 PV) for 114
// VALU instructions; B = 2, 16 heads, 2304 tokens, budget 0.1 (104 GFLOP
// nominal, 312 of MFMA): 290 us = 1.07 PFLOP/s of MFMA, with the split of the
// operands 320 us, against 537 us in the staged kernel (one wave per SIMD,
// every tile split again for every query tile).
//  * LDS: two slots each of a K half (hi and lo plane, 16 KiB) and a V half (8
//    KiB, or 16 KiB with its lo plane): 48 or 64 KiB, so two workgroups share
//    a CU's 160 KiB.
//  * Half step j: wait for K(j + 1) and V(j), issued in the step before; one
//    barrier, which retires every read of K(j) and V(j - 1); issue K(j + 2)
//    and V(j + 1) into their slots; then half j + 1's QK MFMAs with half j's
//    exponentials, half j's PV MFMAs with half j + 1's row max.  (Three slots,
//    the DMAs two steps ahead: 16.7 against 15.8 us at 144 tokens, 32.2 / 31.0
//    at 576, within 1 % above.)
constexpr int kHW = 4;                  // waves per workgroup
constexpr int kHThreads = kHW * 64;
constexpr int kHKBytes = 32 * kSRowBytes;  // a K half: 16 KiB

template <int VDT>
struct HalfShape {
  static constexpr bool kSplitV = VDT == kSplitRows;
  static constexpr int kVBytes = 32 * kD * 2 * (kSplitV ? 2 : 1);
  static constexpr int kVRow = kSplitV ? kSRowBytes : kVRowBytes;
  static constexpr int kRing = 2 * (kHKBytes + kVBytes);
};

// Two P values per dword rounded to MV, and the bf16 rounding of what that leaves.
__device__ __forceinline__ uint32_t pack2_rest(float x, float y, uint32_t hi) {
  const float h0 = __builtin_bit_cast(float, hi << 16);
  const float h1 = __builtin_bit_cast(float, hi & 0xffff0000u);
  return pack2<kBF16>(x - h0, y - h1);
}

// `halves`: the plan's units are items of 256 queries, each run by two
// workgroups (query halves) with the cut index 2 cut + half.
//
// MIXED: tile nfull holds the current rows' last `rest` and the first prior
// rows, as in the 16-bit kernel (seg_attn_pipe_kernel, where the lines of the
// rule are drawn): its DMAs are issued for the lanes of current rows and again
// for the lanes of prior rows.  A last half without keys is left out (kOdd; not
// with 16-bit V beyond the mixed lengths, where its masked half runs).
template <int VDT, bool MIXED>
__global__ __launch_bounds__(kHThreads, 2) void seg_attn_half_kernel(const int32_t* __restrict__ plan_p,
                                                                    const int32_t n_units, const AttnArgs a,
                                                                    const Scalars sc, const int32_t n_qt,
                                                                    const int32_t halves,
                                                                    const RoundSplit split) {
  using Shape = HalfShape<VDT>;
  constexpr bool kSplitV = Shape::kSplitV;
  constexpr int kThreads = kHThreads;
  constexpr int kBM = kHW * 32;
  constexpr int MV = kSplitV ? kBF16 : VDT;
  __shared__ __attribute__((aligned(1024))) uint8_t ring[Shape::kRing];
  __shared__ __attribute__((aligned(16))) int32_t rowtab[3][kBN];
  __shared__ int32_t seg_start[kMaxSegments];
  __shared__ int32_t seg_pref[kMaxSegments + 1];
  __shared__ int32_t merge_turn;
  static_assert(Shape::kRing >= kHW * 32 * kOutPitch, "output staging fits the ring");
  static_assert(kPartialFloats == 66 * kThreads, "partial record layout");

  if (a.append_offsets != nullptr && static_cast<int32_t>(blockIdx.x) >= a.append_first) {
    // a copy block of the fused append, after the attention workgroups
    append_block<kThreads>(a, blockIdx.x - static_cast<uint32_t>(a.append_first), kSRowBytes, Shape::kVRow);
    return;
  }
  // This workgroup's plan unit.  Two workgroups of a 256-query unit sit 8 ids
  // apart: on one XCD, as the plan dealt the unit.
  int32_t uid = static_cast<int32_t>(blockIdx.x);
  int32_t half = 0;
  if (halves != 0) {
    half = (uid >> 3) & 1;
    uid = ((uid >> 4) << 3) + (uid & 7);
  }
  int32_t pu[kPlanInts] = {};
  const bool planned = plan_p != nullptr;
  if (planned) {
    if (uid >= n_units) return;
    const int32_t* src = plan_p + static_cast<int64_t>(uid) * kPlanInts;
#pragma unroll
    for (int i = 0; i < kPlanInts; ++i) pu[i] = src[i];
  }
  const int64_t cap = a.slab_capacity;
  const int H = a.heads;
  const int L = a.cur_len;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform by construction
  const int g = lane >> 5;

  Unit un{0, 0, 1, 0, 0, 0};
  WorkItem w;
  int32_t p0 = 0, p1 = 0;
  bool cut = false;
  if (planned) {
    const int32_t ph = pu[0], pj = pu[1], pcut = pu[4], ppart = pu[5];
    p0 = pu[2];
    p1 = pu[3];
    if (ph < 0 || ph >= H || pj < 0 || pj >= a.batch * n_qt) return;  // not a unit of this launch
    w.h = ph;
    w.b = pj / n_qt;
    w.qt = pj - w.b * n_qt;
    if (halves != 0) {
      w.qt = 2 * w.qt + half;
      if (w.qt * kBM >= L) return;  // no queries in this half (both parts of a cut item leave)
    }
    w.bh = w.b * H + w.h;
    const int32_t c = halves != 0 ? 2 * pcut + half : pcut;
    cut = pcut >= 0 && a.workspace != nullptr && c < a.ws_cuts && ppart >= 0 && ppart < 2;
    un.part = cut ? ppart : 0;
    un.parts = cut ? 2 : 1;
    un.record = cut ? 2 * c : 0;
    un.counter = cut ? c : 0;
    un.arrive = cut && pu[7] != 0 ? 1 : 0;
  } else {
    un = split_unit(split, uid);
    if (split.two == 0) un.item = xcd_item(un.item, a.batch * H, n_qt);
    int32_t* head_rows = reinterpret_cast<int32_t*>(ring);
    w = plan_work<kThreads>(a.seg_starts, a.seg_ends, a.seg_counts, cap, H, a.max_segments, a.batch, n_qt,
                            head_rows, head_rows + kMaxHeads, seg_start, seg_pref, un.item,
                            head_rows + 2 * kMaxHeads, Shape::kRing / 4 - 2 * kMaxHeads);
  }

  // Descriptors: split K rows and V rows of the slab (batch row b) and of the
  // current scale (b, h).
  const int64_t cur_row0 = static_cast<int64_t>(w.bh) * L;
  const int32_t ntc = (L + kBN - 1) / kBN;
  const int32_t nfull = MIXED ? L / kBN : ntc;  // tiles from here on hold prior rows
  const int32_t rest = MIXED ? L - nfull * kBN : 0;
  const u32x4_t dk_prior = make_desc(static_cast<const uint8_t*>(a.slab_k) + w.b * cap * kSRowBytes,
                                     static_cast<uint32_t>(cap * kSRowBytes));
  const u32x4_t dv_prior = make_desc(static_cast<const uint8_t*>(a.slab_v) + w.b * cap * Shape::kVRow,
                                     static_cast<uint32_t>(cap * Shape::kVRow));
  const u32x4_t dk_cur = make_desc(static_cast<const uint8_t*>(a.cur_k) + cur_row0 * kSRowBytes,
                                   static_cast<uint32_t>(L) * kSRowBytes);
  const u32x4_t dv_cur = make_desc(static_cast<const uint8_t*>(a.cur_v) + cur_row0 * Shape::kVRow,
                                   static_cast<uint32_t>(L) * Shape::kVRow);

  // This wave's DMA share of a half: K blocks 4 wave .. + 3 (8 of the hi
  // plane, 8 of the lo plane; 32 key rows x 32 bytes each) and V chunks 2
  // wave, 2 wave + 1 (8 key rows x 128 bytes) of each plane.
  const int k_key = lane & 31;
  const int k_col = (wave >> 1) * (kD * 2) + (wave & 1) * 128 + (lane >> 5) * 16;
  const int lp = lane & 31;
  const int v_key = 16 * (wave >> 1) + 8 * (wave & 1) + 4 * (lp >> 4) + ((lp & 7) >> 1);
  const int v_col = 2 * ((lane >> 5) * 32 + 16 * ((lp >> 3) & 1) + 8 * (lp & 1));
  const uint32_t ring_lds = lds_address(ring);

  // The half's current rows (`cur`) or prior rows; of the mixed tile the lanes
  // of those (zeros past the stream's end).
  auto issue_k_of = [&](int j, auto cur_tag) {
    constexpr bool kCur = decltype(cur_tag)::value;
    const uint32_t dst = ring_lds + (j & 1) * kHKBytes + wave * 4 * 1024;
    const int T = j >> 1, key = (j & 1) * 32 + k_key;
    if (MIXED && T == nfull && (key < rest) != kCur) return;
    int32_t off;
    if constexpr (kCur) {
      off = (j * 32 + k_key) * kSRowBytes + k_col;
    } else {
      const int32_t row = rowtab[(T - nfull) % 3][key];
      off = row < 0 ? kPastEnd : row * kSRowBytes + k_col;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16(kCur ? dk_cur : dk_prior, dst + i * 1024, off + i * 32);
  };
  auto issue_v_of = [&](int j, auto cur_tag) {
    constexpr bool kCur = decltype(cur_tag)::value;
    const uint32_t dst = ring_lds + 2 * kHKBytes + (j & 1) * Shape::kVBytes + wave * 2 * 1024;
    const int T = j >> 1, key = (j & 1) * 32 + v_key;
    if (MIXED && T == nfull && (key < rest) != kCur) return;
    int32_t off;
    if constexpr (kCur) {
      off = (j * 32 + v_key) * Shape::kVRow + v_col;
    } else {
      const int32_t row = rowtab[(T - nfull) % 3][key];
      off = row < 0 ? kPastEnd : row * Shape::kVRow + v_col;
    }
    const u32x4_t d = kCur ? dv_cur : dv_prior;
    dma16(d, dst, off);
    dma16(d, dst + 1024, off + 128);
    if constexpr (kSplitV) {
      dma16(d, dst + 32 * kD * 2, off + kD * 2);
      dma16(d, dst + 32 * kD * 2 + 1024, off + kD * 2 + 128);
    }
  };
  using Cur = std::integral_constant<bool, true>;
  using Prior = std::integral_constant<bool, false>;
  auto has_cur = [&](int j) { return MIXED ? (j >> 1) <= nfull : (j >> 1) < nfull; };
  auto issue_k = [&](int j) {
    if (has_cur(j)) issue_k_of(j, Cur{});
    if ((j >> 1) >= nfull) issue_k_of(j, Prior{});
  };
  auto issue_v = [&](int j) {
    if (has_cur(j)) issue_v_of(j, Cur{});
    if ((j >> 1) >= nfull) issue_v_of(j, Prior{});
  };
  // A unit whose first tile is a current-scale one (every whole item, and a
  // part that starts there) issues it, and Q, before the head's tables load:
  // tables, tile and Q arrive in one round trip.
  const int32_t first = cut ? (p0 < 0 ? 0 : p0) : 0;
  const bool early = planned && first < ntc;
  auto issue_first = [&](int j, auto cur_tag) {
    issue_k_of(j, cur_tag);
    issue_v_of(j, cur_tag);
    issue_k_of(j + 1, cur_tag);
  };
  if (early) issue_first(2 * first, Cur{});

  // Q in two bf16 pieces: B operands of S^T = K Q^T (query row, d = 16ks +
  // 8g .. +7); in flight while the tables load
  const int32_t qrow = w.qt * kBM + wave * 32 + (lane & 31);
  u32x4_t qh[8], ql[8];
  {
    const __amdgpu_buffer_rsrc_t rq = make_rsrc(static_cast<const uint8_t*>(a.q) + cur_row0 * kD * 4,
                                                static_cast<uint32_t>(L * kD * 4));
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      load8_split(rq, qrow < L ? (qrow * kD + ks * 16 + g * 8) * 4 : -1, qh[ks], ql[ks]);
  }
  if (planned)
    load_head_segments<kThreads>(a.seg_starts, a.seg_ends, a.seg_counts, cap, a.max_segments, w, seg_start,
                                 seg_pref);
  const int32_t R = w.R;
  const int32_t ntiles = MIXED ? (L + R + kBN - 1) / kBN : (R + kBN - 1) / kBN + ntc;
  int32_t parts = un.parts;
  int32_t tb = 0, te = ntiles;
  if (planned) {
    if (cut) {
      tb = p0 < 0 ? 0 : (p0 > ntiles ? ntiles : p0);
      te = p1 < tb ? tb : (p1 > ntiles ? ntiles : p1);
    }
  } else {
    // as in the 16-bit kernel: a part needs min_part tiles, parts past
    // the count leave at once
    parts = ntiles / split.min_part;
    parts = parts < 1 ? 1 : (parts < un.parts ? parts : un.parts);
    if (un.part >= parts) return;
    tb = un.part * ntiles / parts;
    te = (un.part + 1) * ntiles / parts;
  }
  if (tb >= te) {
    // a planned part with no key tiles (a plan that does not match these
    // tables): its record is empty -- zero weight in the merge
    wait_vmcnt<0>();  // an early tile lands before the LDS is used again
    f32x16_t none[4] = {};
    merge_parts<kF32, kThreads>(a, sc, un, parts, none, -1e30f, 0.f, w, qrow, L, H, g, merge_turn,
                                ring + wave * 32 * kOutPitch);
    return;
  }

  auto valid_of = [&](int T) {
    if constexpr (MIXED) return min(kBN, L + R - T * kBN);
    return T < ntc ? min(kBN, L - T * kBN) : min(kBN, R - (T - ntc) * kBN);
  };
  int cur_seg = 0;
  auto fill = [&](int T) {  // wave 0: row table of tile T (one with prior rows)
    if (T >= nfull && T < te)
      fill_rowtab<1>(T - nfull, rowtab[(T - nfull) % 3], cur_seg, w.nseg, R, seg_start, seg_pref, -1, rest);
  };

  const int j0 = 2 * tb;
  constexpr bool kOdd = MIXED || kSplitV;
  const int jend = 2 * te - (kOdd && valid_of(te - 1) <= 32 ? 1 : 0);
  if (wave == 0) {
    fill(tb);
    fill(tb + 1);
  }
  __syncthreads();
  if (!early && has_cur(j0)) issue_first(j0, Cur{});
  if (tb >= nfull) issue_first(j0, Prior{});
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    qh[ks] ^= sc.q_sign;
    ql[ks] ^= sc.q_sign;
  }

  f32x16_t oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) oacc[i] = f32x16_t{};
  float m_run = -1e30f;
  float l_run = 0.f;

  // S^T of half j from its slot
  auto qk = [&](f32x16_t& s, int j) {
    const uint8_t* kst = ring + (j & 1) * kHKBytes + lane * 16;
    s = f32x16_t{};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const u32x4_t kh = *reinterpret_cast<const u32x4_t*>(kst + ks * 1024);
      const u32x4_t kl = *reinterpret_cast<const u32x4_t*>(kst + (8 + ks) * 1024);
      s = mfma32<kBF16>(kh, qh[ks], s);
      s = mfma32<kBF16>(kh, ql[ks], s);
      s = mfma32<kBF16>(kl, qh[ks], s);
    }
  };
  // O^T += V^T P^T over half j's keys
  auto pv = [&](const f32x16_t& s, int j) {
    const uint8_t* vst = ring + 2 * kHKBytes + (j & 1) * Shape::kVBytes + lane * 8;
#pragma unroll
    for (int ul = 0; ul < 2; ++ul) {
      u32x4_t ph, pl;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ph[i] = pack2<MV>(s[8 * ul + 2 * i], s[8 * ul + 2 * i + 1]);
        if constexpr (kSplitV) pl[i] = pack2_rest(s[8 * ul + 2 * i], s[8 * ul + 2 * i + 1], ph[i]);
      }
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const uint8_t* const blk = vst + ul * 4096 + (db >> 1) * 1024 + (db & 1) * 512;
        const u32x2_t lo = ds_read_tr(blk);
        const u32x2_t hi = ds_read_tr(blk + 2048);
        const u32x4_t vh = {lo[0], lo[1], hi[0], hi[1]};
        oacc[db] = mfma32<MV>(vh, ph, oacc[db]);
        if constexpr (kSplitV) {
          const u32x2_t lo2 = ds_read_tr(blk + 32 * kD * 2);
          const u32x2_t hi2 = ds_read_tr(blk + 32 * kD * 2 + 2048);
          const u32x4_t vl = {lo2[0], lo2[1], hi2[0], hi2[1]};
          oacc[db] = mfma32<MV>(vh, pl, oacc[db]);
          oacc[db] = mfma32<MV>(vl, ph, oacc[db]);
        }
      }
    }
  };
  auto masked_max = [&](f32x16_t& s, int j) {
    float mx = half_max(s);
    asm volatile("" : "+v"(mx));
    const int v = valid_of(j >> 1);
    if (v < 32 * ((j & 1) + 1)) {
      mask_half(s, j & 1, v, g);
      mx = half_max(s);
    }
    return mx;
  };

  // Prologue: every issued half landed; S of the first half and its max.
  wait_vmcnt<0>();
  __syncthreads();
  f32x16_t sa, sb;
  qk(sa, j0);
  move_max(oacc, m_run, l_run, masked_max(sa, j0), sc.c, sc.thresh);

  // Half step j: scur = S(j) (max applied), snext receives S(j + 1) unless j
  // is the item's last half.
  auto step = [&](auto more_tag, f32x16_t& scur, f32x16_t& snext, int j) {
    constexpr bool kMore = decltype(more_tag)::value;
    wait_vmcnt<0>();  // this wave's share of K(j + 1) and V(j)
    __syncthreads();
    if constexpr (kMore) {
      if (j + 2 < jend) issue_k(j + 2);
      issue_v(j + 1);
    }
    // the table of the tile whose K is first issued in the next step
    if (wave == 0 && (j & 1) != 0) fill((j + 3) >> 1);
    if constexpr (kMore) qk(snext, j + 1);
    exp_half(scur, m_run, sc.c, l_run);
    pv(scur, j);
    if constexpr (kMore) {
      asm volatile("" : "+v"(l_run));
      move_max(oacc, m_run, l_run, masked_max(snext, j + 1), sc.c, sc.thresh);
    }
  };
  using More = std::integral_constant<bool, true>;
  using Last = std::integral_constant<bool, false>;
  int j = j0;
  for (; j + 2 < jend; j += 2) {
    step(More{}, sa, sb, j);
    step(More{}, sb, sa, j + 1);
  }
  if (!kOdd || j + 1 < jend) {
    step(More{}, sa, sb, j);
    ++j;
  } else {
    sb = sa;  // an odd count: one Last step serves both (two spill registers)
  }
  step(Last{}, sb, sa, j);

  if (parts == 1) {
    if (a.out_dtype != kF32 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0) {
      __syncthreads();  // every wave is past its last half: the ring is free
      uint8_t* const stage = ring + wave * 32 * kOutPitch;
      const int32_t qrow0 = w.qt * kBM + wave * 32;
      if (a.out_dtype == kF16)
        write_output_lds<kF16>(oacc, m_run, l_run, sc.c, a.out, a.lse, w.b, w.h, qrow0, L, H, w.bh, lane, stage);
      else
        write_output_lds<kBF16>(oacc, m_run, l_run, sc.c, a.out, a.lse, w.b, w.h, qrow0, L, H, w.bh, lane, stage);
    } else {
      write_output(oacc, m_run, l_run, sc.c, a.out, a.lse, w.b, w.h, qrow, L, H, w.bh, g, a.out_dtype);
    }
    return;
  }
  merge_parts<kF32, kThreads>(a, sc, un, parts, oacc, m_run, l_run, w, qrow, L, H, g, merge_turn,
                              ring + wave * 32 * kOutPitch);
}

template <int VDT>
hipError_t launch_half(const AttnArgs& a, const Scalars& s, hipStream_t st, int32_t plan_queries) {
  const int32_t n_qt = (a.cur_len + 127) / 128;
  const int64_t items = static_cast<int64_t>(a.batch) * a.heads * n_qt;
  if (items <= 0) return hipSuccess;
  if (items > 0x3fffffffLL) return hipErrorInvalidConfiguration;
  int device = 0;
  const int32_t slots = a.workspace != nullptr && hipGetDevice(&device) == hipSuccess ? split_slots(device) : 0;
  RoundSplit split{static_cast<int32_t>(items), 0, 0, 0, 1, 0};
  if (slots > 0 && a.workspace_bytes >= split_workspace_bytes(slots))
    split = round_split(static_cast<int32_t>(items), slots, (a.cur_len + kBN - 1) / kBN);
  AttnArgs b = a;
  b.ws_cuts = 0;
  if (a.workspace != nullptr && a.workspace_bytes > kCounterBytes) {
    const int64_t by_records = (a.workspace_bytes - kCounterBytes) / (2LL * kPartialFloats * 4);
    b.ws_cuts = static_cast<int32_t>(by_records < kMaxCounters ? by_records : kMaxCounters);
  }
  const bool halves = a.plan != nullptr && plan_queries == kSBM;
  int64_t grid = a.plan != nullptr ? a.plan_units : split_units(split);
  if (halves) grid = (grid + 7) / 8 * 16;
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  const int32_t units = b.plan != nullptr ? b.plan_units : 0;
  const int32_t tiles = halves ? (a.cur_len + kSBM - 1) / kSBM : n_qt;
  const int64_t copies = a.append_offsets != nullptr ? append_blocks(a.batch, a.heads, a.cur_len) : 0;
  if (grid + copies > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  b.append_first = static_cast<int32_t>(grid);
  const dim3 blocks(static_cast<uint32_t>(grid + copies));
  if (a.cur_len % kBN != 0 && a.cur_len < kMixedBelow)
    seg_attn_half_kernel<VDT, true><<<blocks, kHThreads, 0, st>>>(b.plan, units, b, s, tiles, halves ? 1 : 0, split);
  else
    seg_attn_half_kernel<VDT, false><<<blocks, kHThreads, 0, st>>>(b.plan, units, b, s, tiles, halves ? 1 : 0, split);
  return hipGetLastError();
}

// Whether a call on split K rows with 16-bit V runs as 128-query workgroups
// (seg_attn_half_kernel; a plan's 256-query units as two halves each) instead
// of 256-query ones.  The 8-wave form is the faster one once every CU has its
// fill of it, the halves before that: they spread over twice the workgroups, a
// last tile of at most 128 queries costs half, a call without a plan cuts its
// items in two (one image pair, 16 heads, not planned, us, halves / 8 waves at
// 144, 576, 1024, 1600, 2304, 4096 tokens: 17.2 / 20.4, 37.0 / 47.2, 58.5 / 96.9,
// 105.7 / 126, 203 / 229, 613 / 587), and their launch takes the append, which
// follows the 8-wave one as a launch of its own.  16 heads, a tenth retained /
// heads of uneven lengths, planned, K split by the producer, us, halves : 8 waves
// by 256-query items:
// * no append, up to one half per CU: 64 items (1024 tokens) 34.8 : 43.6 / 42.8 :
//   56.6, 112 (1600) 63.7 : 62.0 / 74.9 : 80.9, 128 (B=2, 1024) 50.8 : 52.2 / 62.1 :
//   63.8.  Above, some CUs share two halves while others have one: 144 (2304)
//   115.9 : 105.2 / 129 : 133, 192 (B=2, 1296) 90.9 : 82.9 / 100.4 : 98.0, 224 (B=2,
//   1600) 109.7 : 101.7 / 127.2 : 130.3, 256 (4096) 283 : 259 / 331 : 317.
// * with the append, up to two items per CU (where every head appends) and
//   2560 tokens: 192 (B=2, 1296) 92.1 : 92.7 / 101.7 : 109.1, 192 (B=3, 1024)
//   77.0 : 81.1 / 90.6 : 97.3, 224 111.5 : 115.2 / 130 : 144, 288 (B=2, 2304) 218 : 222 /
//   235 : 239, 432 (B=3, 2304) 314 : 318 / 352 : 351, but 176 (2704) 169 : 155 / 174 :
//   180, 256 (4096) 286 : 275 / 333 : 332, and 660 (B=2, 30 heads, 2704) 522 : 513.
// Without a plan: below two 256-query items per CU.  And where half tiles save
// at least an eighth of the padded queries (576 tokens, 768 items: 135 / 143 us;
// 1600 tokens save 7 %: 771 / 753).
constexpr int32_t kHalvesAppendLen = 2560;
bool split_in_halves(const AttnArgs& a) {
  int device = 0;
  const int64_t cus = hipGetDevice(&device) == hipSuccess ? split_slots(device) / 2 : 0;
  const int64_t t256 = (static_cast<int64_t>(a.cur_len) + kSBM - 1) / kSBM;
  const int64_t t128 = (static_cast<int64_t>(a.cur_len) + 127) / 128;
  const int64_t items = static_cast<int64_t>(a.batch) * a.heads * t256;
  if (a.plan == nullptr) {
    if (items < 2 * cus) return true;
  } else if (a.append_offsets != nullptr && a.cur_len <= kHalvesAppendLen) {
    if (items <= 2 * cus) return true;
  } else if (2 * items <= cus) {
    return true;
  }
  return 8 * t128 <= 7 * 2 * t256;
}

template <int VDT>
hipError_t launch(const AttnArgs& a, const Scalars& s, hipStream_t st) {
  const int32_t n_qt = (a.cur_len + kSBM - 1) / kSBM;
  const int64_t items = static_cast<int64_t>(a.batch) * a.heads * n_qt;
  if (items <= 0) return hipSuccess;
  if (items > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  AttnArgs b = a;
  b.ws_cuts = 0;
  if (a.workspace != nullptr && a.workspace_bytes > kCounterBytes) {
    const int64_t by_records = (a.workspace_bytes - kCounterBytes) / (2LL * 66 * kSThreads * 4);
    b.ws_cuts = static_cast<int32_t>(by_records < kMaxCounters ? by_records : kMaxCounters);
  }
  const int64_t grid = a.plan != nullptr ? a.plan_units : items;
  if (grid <= 0) return hipSuccess;
  seg_attn_split_kernel<VDT><<<dim3(static_cast<uint32_t>(grid)), kSThreads, 0, st>>>(
      b.plan, b.plan != nullptr ? static_cast<int32_t>(grid) : 0, b, s, n_qt);
  return hipGetLastError();
}

}  // namespace

bool attention_split_supported(const AttnArgs& a) {
  const bool v16 = a.v_dtype == kBF16 || a.v_dtype == kF16;
  return a.q_dtype == kF32 && a.k_dtype == kSplitRows && v16 && a.heads <= kMaxHeads &&
         a.qk_dot_mode != kDotFp32 && a.value_dot_mode != kDotFp32;
}

// The append rides in the 128-query form's launch (a layer's early and middle
// scales, where a launch of its own costs 2-3 us) and follows the 256-query one.
hipError_t launch_attention_split(const AttnArgs& a, const attn::Scalars& s, hipStream_t stream) {
  if (a.v_dtype == kSplitRows) {  // only from hkv_segmented_attention_split: plans of 128-query items
    if (a.q_dtype != kF32 || a.k_dtype != kSplitRows) return hipErrorInvalidValue;
    return launch_half<kSplitRows>(a, s, stream, 128);
  }
  if (!attention_split_supported(a)) return hipErrorInvalidValue;
  if (split_in_halves(a))
    return a.v_dtype == kBF16 ? launch_half<kBF16>(a, s, stream, kSBM) : launch_half<kF16>(a, s, stream, kSBM);
  const hipError_t e = a.v_dtype == kBF16 ? launch<kBF16>(a, s, stream) : launch<kF16>(a, s, stream);
  return e != hipSuccess || a.append_offsets == nullptr ? e : launch_append(a, stream);
}

hipError_t launch_split_operands(SplitOperands o, bool with_v, hipStream_t stream) {
  const int64_t cur_blocks = (o.cur_rows + kSplitCurRows - 1) / kSplitCurRows;
  o.slab_chunks = o.max_segments > 0 ? (o.slab_capacity + kSplitSlabRows - 1) / kSplitSlabRows : 0;
  o.slab_blocks = o.batch * o.slab_chunks;
  const int64_t blocks = cur_blocks + o.slab_blocks;
  if (blocks <= 0) return hipSuccess;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  split_operands_kernel<<<dim3(static_cast<uint32_t>(blocks), with_v ? 2 : 1), 256, 0, stream>>>(o);
  return hipGetLastError();
}

hipError_t launch_split_rows(const float* src, void* dst, int64_t rows, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const int64_t blocks = (rows * 16 + 255) / 256;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  split_rows_kernel<<<dim3(static_cast<uint32_t>(blocks)), 256, 0, stream>>>(src, static_cast<uint8_t*>(dst),
                                                                              rows);
  return hipGetLastError();
}

int32_t attention_item_queries(const AttnArgs& a) { return attention_split_supported(a) ? kSBM : 128; }

}  // namespace hkv
