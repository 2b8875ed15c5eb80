// Paged decode attention with a fixed reduction order (gfx950).
//
// Behaviour follows paged_attn.py:21-114: one query token per request, GQA groups of
// G = H / KV query heads per KV head, keys cut into fixed segments of `split` keys whose
// count NS = cdiv(max_len, split) is fixed by the model length, segment partials
// (m, l, acc) merged in segment order. The floating-point order depends only on the
// request's own length and the constants (split, blk, waves): never on the batch, on the
// other requests, or on where the pages sit in memory.
//
// Kernel shape (MI355X-first, not a translation of the Triton kernel):
//  * a segment is cut into units of 64 keys (one exception: ONE_UNIT); a wave runs an online softmax
//    over one unit at a time and merges its units (wave, wave + NW, ...) in order, the NW waves of
//    the segment are merged in order, then the segments. A workgroup computes a whole segment of
//    (request b, KV head g); where that leaves most CUs idle (a few requests), it computes NW units
//    only and writes their partials, which a second kernel merges in the same order: the same bits;
//  * S = K q^T on bf16 matrix cores (v_mfma_f32_16x16x32_bf16): rows are 16 keys of a tile,
//    columns the G query heads of the group (bf16 x bf16 products are exact in fp32);
//  * online softmax in base 2 on the hardware v_exp_f32, state per head kept in fp32;
//  * P V on the vector ALU in fp32: each lane owns D/16 output dims for a quarter of the
//    tile's keys, p arrives by row broadcasts (DPP), V is read as 16-byte rows. fp32 p times bf16
//    v keeps all 24 bits of p, which is what the reference's hi/lo bf16 split of p
//    (paged_attn.py:63-65) approximates with 2 x 8 bits on bf16 tensor cores;
//  * K and V are read with nontemporal loads: every cache byte is read once per step, and on
//    gfx950 a stream of permuted 8 KiB pages reads at ~6.6 TB/s that way against ~5.8 TB/s
//    with the default cache policy (same pages, same lanes; the load policy is all that
//    differs).
//
// What bounds it: HBM on large grids; on small ones the latency of a wave's tiles. A wave keeps
// a ring of tiles in flight (32 KiB of K and V at D = 128, in registers), each refilled when its
// tile has been used, also across units, so neither K nor V is waited for in the steady state;
// exchanges between lane rows are lane swaps and DPP operands instead of LDS round trips; where
// a page holds whole tiles, a row address is a scalar base and a lane offset. Measured at
// H32/KV8/D128, page 16, event-timed calls, us, K then V read per tile with LDS
// exchanges -> this: one request of 16384 keys 88.5 -> 21.2 (units; whole segments 35.3), of 1024
// 44.5 -> 11.2; 4 of 16384 97.0 -> 49.7 (2.8 -> 5.4 TB/s); 32 of 1024 49.6 -> 26.1; 64 of 8192
// 342.6 -> 339.7 (6.3 TB/s), with lengths spread over 4096..8192 298.8 -> 276.1; 256 of 1024 at
// H16/KV2/D256, page 528: 186.5 -> 113.0. The units also shorten the fp32 sums: the error against
// float64 fell by 18 % over 27 shapes of 64 to 16384 keys (largest 2.99e-7 -> 2.40e-7).
// Arithmetic is compiled with -ffp-contract=off; every fused multiply-add is written
// explicitly, so the order is the one in the source.

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

struct PagedParams {
  const uint16_t* q;
  int64_t sqt, sqh;
  const uint16_t* kc;
  int64_t skb, skp, skh;
  const uint16_t* vc;
  int64_t svb, svp, svh;
  const int32_t* bt;
  int64_t sbt;
  const int32_t* sl;
  float scale_log2;  // softmax scale * log2(e)
  int32_t split;     // keys per segment (multiple of 16)
  int32_t ns;        // segments per request in the grid (the caller's length bound may trim it)
  int32_t ns_model;  // segments the model's maximum length fixes: NS = cdiv(max_len, split)
  int32_t H, KV;
  int32_t bs;        // page size (tokens per block)
  int32_t bs_shift;  // log2(bs) when bs is a power of two, else -1
  int64_t n;
  const int32_t* n_live;  // device count of requests to compute (<= n), or null for all n
  int32_t units;   // units of kUnit keys in a segment
  int32_t slices;  // workgroups of a segment when its units are computed apart
  int32_t slice_units;  // units of such a workgroup
  float* mp;  // [n][H][ns], or [n][H][ns][units]
  float* lp;  // as mp
  float* ap;  // as mp, [D] each
  void* out;
  int64_t sot, soh;
  int32_t out_dtype;
};

constexpr float kNegInf = -__builtin_huge_valf();
// Where a unit's running maximum starts: below every finite score, so that the first tile replaces it,
// and finite, so that keys scoring -inf weigh exp2(-inf - m) = 0 also where nothing else has been seen
// (-inf - -inf would be NaN). Such a unit's state is (kLowest, 0, 0), which adds 0 to any merge.
constexpr float kLowest = -3.402823466e38f;  // -FLT_MAX

__device__ inline float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// Fixed-order merge of a softmax state (m, l, a) with another (ms, ls, as_)
// (paged_attn.py:84-93, base-2 logits). A state with m == -inf contributes exactly 0.
__device__ inline void merge_state(float& m, float& l, float& a, float ms, float ls, float as_) {
  const float mn = fmaxf(m, ms);
  const float c_old = (m == kNegInf) ? 0.0f : exp2_hw(m - mn);
  const float c_new = (ms == kNegInf) ? 0.0f : exp2_hw(ms - mn);
  l = fmaf(l, c_old, ls * c_new);
  a = fmaf(a, c_old, as_ * c_new);
  m = mn;
}

__device__ inline int32_t page_of(const PagedParams& p, int key) {
  return p.bs_shift >= 0 ? (key >> p.bs_shift) : (int32_t)((uint32_t)key / (uint32_t)p.bs);
}

// Element offset of `key`'s row in a cache with block stride sb and token stride sp. The
// segment's block-table entries sit in LDS (pages[i] = block_table[b][blk0 + i]), so the K/V
// address never waits on a global load of the table.
__device__ inline int64_t page_offset(const PagedParams& p, const int32_t* pages, int blk0, int key, int64_t sb,
                                      int64_t sp) {
  const int32_t blk = page_of(p, key);
  const int32_t off = key - blk * p.bs;
  return (int64_t)pages[blk - blk0] * sb + (int64_t)off * sp;
}

template <int D>
struct DimTraits {
  static constexpr int kQkSteps = D / 32;  // MFMA K steps of 32 over the head dim
  static constexpr int kDpl = D / 16;      // output dims per lane in P V
};

// Keys of one unit: a wave's online softmax runs over one unit and its state is then merged into
// the wave's running state, so that units can also be computed apart and merged later.
constexpr int kUnit = 64;

// Exchanges between the four 16-lane rows of a wave on the vector ALU (gfx950 lane swaps), in
// place of ds_bpermute round trips through the LDS pipe. The fp32 pairs come back as
// {x of the lower row or half, x of the upper}, for both sides.
__device__ inline void swap32(float& a, float& b) {  // a's upper half <-> b's lower half
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ inline void swap16(float& a, float& b) {  // a's odd rows <-> b's even rows
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ inline float rows_max(float v) {
  float a = v, b = v;
  swap16(a, b);
  v = fmaxf(a, b);
  a = v, b = v;
  swap32(a, b);
  return fmaxf(a, b);
}
__device__ inline float rows_sum(float v) {
  float a = v, b = v;
  swap16(a, b);
  v = a + b;
  a = v, b = v;
  swap32(a, b);
  return a + b;
}
// Lane H of the caller's 16-lane row, for every lane of the row (a DPP operand, no LDS).
template <int H>
__device__ inline float row_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + H, 0xf, 0xf, false));
}

template <int N, typename F, int I = 0>
__device__ inline void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, F, I + 1>(static_cast<F&&>(f));
  }
}

// 16-byte (8-byte for D = 64) pieces of V a lane reads per key, raw.
template <int D>
struct VRaw {
  static constexpr int kWords = D / 32;
  uint32_t w[kWords];
};
template <int D>
__device__ inline VRaw<D> load_v(const uint16_t* p) {
  VRaw<D> r;
  if constexpr (D == 64) {
    const v2u32 u = __builtin_nontemporal_load(reinterpret_cast<const v2u32*>(p));
    r.w[0] = u.x;
    r.w[1] = u.y;
  } else {
#pragma unroll
    for (int c = 0; c < D / 128; ++c) {
      const v4u32 u = __builtin_nontemporal_load(reinterpret_cast<const v4u32*>(p + 8 * c));
      r.w[4 * c] = u.x;
      r.w[4 * c + 1] = u.y;
      r.w[4 * c + 2] = u.z;
      r.w[4 * c + 3] = u.w;
    }
  }
  return r;
}

// Tiles of 16 keys whose K and V loads a wave has in flight when AHEAD: at D = 128 four tiles, 128
// VGPRs and 32 KiB; at D = 256 two, the same, or one (64 VGPRs) where the accumulators of 4 or 8 heads
// need the registers (4 heads keep two waves a SIMD); at D = 64 four, 64 VGPRs and 16 KiB (a ring
// is at most a unit's tiles). 8 heads of 128 dims on whole segments (260 VGPRs) and 2 of 256 (260-268)
// leave one wave a SIMD and are still faster than without the ring at more waves: 64 requests of
// 4096 to 8192 keys, 4 KV heads, D = 128, G = 8 220.8 -> 183.6 us, 256 of 512 to 1024 109.2 -> 102.2;
// 8 KV heads, D = 256, G = 2, 64 of 1024 to 2048 170.1 -> 163.7, 256 of 512 to 1024 325.1 -> 308.8.
template <int D, int G>
constexpr int ahead_tiles() {
  return D == 256 ? (G >= 4 ? 1 : 2) : 4;
}

// UNITS: a workgroup computes a slice of a segment (slice_units consecutive units, the waves
// taking them in turn) and writes each unit's partial (paged_merge_units_kernel merges them).
// Otherwise it computes a whole segment, each wave merging its units (wave, wave + NW, ...) in
// order, then the waves in order. Both do the same operations on the same values in the same order.
template <int D, int G, int TPG, int NW, bool UNITS, bool AHEAD, bool ALIGNED>
__global__ __launch_bounds__(64 * NW) void paged_partial_kernel(PagedParams p) {
  static_assert(G >= 1 && G <= 16, "GQA group must fit the 16 MFMA columns");
  static_assert(!AHEAD || TPG == 1, "loads ahead are written for one tile a step");
  static_assert(AHEAD || !ALIGNED, "page-aligned tiles are written for loads ahead");
  constexpr int QS = DimTraits<D>::kQkSteps;
  constexpr int DPL = DimTraits<D>::kDpl;
  constexpr int FL = G * DPL;  // accumulators of a lane
  constexpr int QF = FL / 4;   // and the quarter of them its row owns once the rows are summed
  // 8 waves of 128 accumulators a lane and two tiles a step (8 heads of 256 dims at 32 keys) have no
  // registers for a running state beside a unit's: there a wave's whole share is one unit. 64 requests
  // of 2048 to 4096 keys, us: 278 before there were units, 367 with a merge per 64 keys (113 VGPRs
  // spilled), 290 this way.
  constexpr bool ONE_UNIT = !AHEAD && FL >= 128 && TPG == 2 && NW == 8;
  __shared__ float s_m[NW][G];
  __shared__ float s_l[NW][G];
  __shared__ float s_acc[NW][G][D];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar loop control
  const int col = lane & 15;  // S layout: head column / PV layout: dim chunk
  const int row = lane >> 4;  // S layout: key quad / PV layout: key quarter

  const int64_t per_seg = p.n * p.KV;
  const int part = (int)(blockIdx.x / per_seg);  // segment, or slice of a segment
  const int s = UNITS ? part / p.slices : part;
  const int64_t rem = blockIdx.x % per_seg;
  const int b = (int)(rem / p.KV);
  const int g = (int)(rem % p.KV);
  if (p.n_live != nullptr && b >= *p.n_live) return;  // not a live request: nothing read or written

  const int L = p.sl[b];

  // Segments the request needs, capped at the model's NS as the fixed grid caps them. A grid
  // trimmed by the caller's bound on the batch's lengths covers every request within that
  // bound with the same segments (the same bits); a longer request gets NaN rows, written by
  // its first workgroups, instead of a sum over fewer keys.
  const int need = min((L + p.split - 1) / p.split, p.ns_model);
  if (need > p.ns) {
    if (part == 0)
      for (int idx = threadIdx.x; idx < G * D; idx += 64 * NW)
        store_f32_as(p.out, p.out_dtype, (int64_t)b * p.sot + (int64_t)(g * G + idx / D) * p.soh + idx % D,
                     __builtin_nanf(""));
    return;
  }
  // Keys [start, end) of this workgroup; its units start there.
  int start = s * p.split;
  int end = min(start + p.split, L);
  int unit0 = 0;  // index of its first unit in the segment
  if constexpr (UNITS) {
    unit0 = (part % p.slices) * p.slice_units;
    start += unit0 * kUnit;
    end = min(end, start + p.slice_units * kUnit);
  }
  if (start >= end) return;  // past the end: contributes exactly 0, never read

  // The segment's block-table entries, staged once into LDS (dynamic shared memory sized
  // split / bs + 2 entries by the launcher).
  extern __shared__ int32_t s_pages[];
  const int blk0 = page_of(p, start);
  const int npg = page_of(p, end - 1) - blk0 + 1;
  for (int i = threadIdx.x; i < npg; i += 64 * NW) s_pages[i] = p.bt[(int64_t)b * p.sbt + blk0 + i];

  // q as the B operand: column = head (g*G + col), 8 dims per lane per MFMA step.
  v8bf qf[QS];
  {
    const uint16_t* qrow = p.q + (int64_t)b * p.sqt + (int64_t)(g * G + (col < G ? col : 0)) * p.sqh;
#pragma unroll
    for (int i = 0; i < QS; ++i) {
      v8u16 raw = *reinterpret_cast<const v8u16*>(qrow + 32 * i + 8 * row);
      if (col >= G) raw = v8u16{0, 0, 0, 0, 0, 0, 0, 0};
      qf[i] = __builtin_bit_cast(v8bf, raw);
    }
  }
  __syncthreads();

  const int64_t khead = (int64_t)g * p.skh;
  const int64_t vhead = (int64_t)g * p.svh;
  auto krow_of = [&](int tile_key) {  // lane col -> key, 8 dims per lane per step
    const int key = min(tile_key + col, end - 1);
    return p.kc + page_offset(p, s_pages, blk0, key, p.skb, p.skp) + khead + 8 * row;
  };
  auto vrow_of = [&](int tile_key, int j) {
    const int key = min(tile_key + 4 * row + j, end - 1);
    return p.vc + page_offset(p, s_pages, blk0, key, p.svb, p.svp) + vhead + col * DPL;
  };
  auto load_k = [&](const uint16_t* krow, int i) {
    return __builtin_nontemporal_load(reinterpret_cast<const v8u16*>(krow + 32 * i));
  };

  float m_tot = kNegInf, l_tot = 0.0f;  // the wave's units so far, per head column (S layout)
  float a_tot[QF];                       // the flat accumulators [row * QF, row * QF + QF)
#pragma unroll
  for (int i = 0; i < QF; ++i) a_tot[i] = 0.0f;

  // Tiles in flight per wave when AHEAD: slot (tile % PT) of the ring holds one tile's K and V.
  constexpr int PT = AHEAD ? ahead_tiles<D, G>() : 1;
  constexpr int kTiles = kUnit / 16;
  static_assert(kTiles % PT == 0, "a unit's tiles walk the ring whole");
  v8u16 kr[PT][QS];
  VRaw<D> vr[PT][4];
  // ALIGNED (pages of whole 16-key tiles): a tile's page comes from one LDS read per unit (lane t
  // reads tile t's entry) and the row addresses are a scalar base and one lane offset per cache.
  const uint32_t koff_lane = ALIGNED ? (uint32_t)((col * p.skp + 8 * row) * 2) : 0u;
  const uint32_t voff_lane = ALIGNED ? (uint32_t)((4 * row * p.svp + col * DPL) * 2) : 0u;
  struct TilePages {
    int32_t page, off;  // lane t: tile t's block-table entry and its first row in the page
  };
  auto unit_pages = [&](int u) {  // a tile past the end takes the last key's row
    const int key = min(start + u * kUnit + 16 * (lane & (kTiles - 1)), end - 1);
    const int pg = page_of(p, key);
    return TilePages{s_pages[pg - blk0], key - pg * p.bs};
  };
  auto issue = [&](int slot, int tile_key, const TilePages& pages, int t) {  // keys past the end repeat the last key's rows
    if constexpr (ALIGNED) {
      const int64_t off0 = __builtin_amdgcn_readlane(pages.off, t);
      const int64_t page = __builtin_amdgcn_readlane(pages.page, t);
      const char* kb = reinterpret_cast<const char*>(p.kc + page * p.skb + off0 * p.skp + khead);
      const char* vb = reinterpret_cast<const char*>(p.vc + page * p.svb + off0 * p.svp + vhead);
      uint32_t koff = koff_lane, voff[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) voff[j] = voff_lane + (uint32_t)(j * p.svp * 2);
      const int last = max(end - 1 - tile_key, 0);  // the tile's last live key
      if (last < 15) {
        koff = (uint32_t)((min(col, last) * (int)p.skp + 8 * row) * 2);
#pragma unroll
        for (int j = 0; j < 4; ++j) voff[j] = (uint32_t)((min(4 * row + j, last) * (int)p.svp + col * DPL) * 2);
      }
#pragma unroll
      for (int i = 0; i < QS; ++i)
        kr[slot][i] = __builtin_nontemporal_load(reinterpret_cast<const v8u16*>(kb + koff + 64 * i));
#pragma unroll
      for (int j = 0; j < 4; ++j) vr[slot][j] = load_v<D>(reinterpret_cast<const uint16_t*>(vb + voff[j]));
    } else {
      const uint16_t* krow = krow_of(tile_key);
#pragma unroll
      for (int i = 0; i < QS; ++i) kr[slot][i] = load_k(krow, i);
#pragma unroll
      for (int j = 0; j < 4; ++j) vr[slot][j] = load_v<D>(vrow_of(tile_key, j));
    }
    asm volatile("" ::: "memory");  // issued here, ahead of the arithmetic below
  };
  TilePages pages = {0, 0};  // ALIGNED: of the unit whose loads are issued

  // One unit of this wave; `next` (AHEAD): the wave has a further unit, NW units on.
  auto unit = [&](int u, auto next) {
    const int ubase = start + u * kUnit;
    const int uend = ONE_UNIT ? end : min(ubase + kUnit, end);
    float m_run = kLowest, l_run = 0.0f;  // per head column (S layout)
    float acc[FL];                         // PV layout: head x owned dims
#pragma unroll
    for (int i = 0; i < FL; ++i) acc[i] = 0.0f;

    // One group of TPG tiles at kbase: k_at(t, i) and v_at(t, j) give its K and V.
    auto group = [&](int kbase, auto&& k_at, auto&& v_at) {
      float sc[TPG][4];
#pragma unroll
      for (int t = 0; t < TPG; ++t) {
        v4f c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < QS; ++i)
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, k_at(t, i)), qf[i], c, 0, 0, 0);
        // c[r] = S[key kbase + 16t + 4*row + r][head col]
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int kk = kbase + 16 * t + 4 * row + r;
          sc[t][r] = (kk < uend) ? c[r] * p.scale_log2 : kNegInf;
        }
      }
      // Online softmax update for this group, fixed order.
      float mx = kNegInf;
#pragma unroll
      for (int t = 0; t < TPG; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[t][r]);
      const float m_new = fmaxf(m_run, rows_max(mx));
      const float alpha = exp2_hw(m_run - m_new);  // m_run == kLowest -> 0, or nothing to rescale
      float psum = 0.0f;
#pragma unroll
      for (int t = 0; t < TPG; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[t][r] = exp2_hw(sc[t][r] - m_new);
          psum += sc[t][r];
        }
      l_run = fmaf(l_run, alpha, rows_sum(psum));
      m_run = m_new;

      // P V. Rescale the owned accumulators by each head's alpha (held by lane col == h).
      static_for<G>([&](auto h) {
        const float ah = row_lane<h>(alpha);
#pragma unroll
        for (int d = 0; d < DPL; ++d) acc[h * DPL + d] = acc[h * DPL + d] * ah;
      });
#pragma unroll
      for (int t = 0; t < TPG; ++t) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const VRaw<D> raw = v_at(t, j);
          float v[DPL];
#pragma unroll
          for (int e = 0; e < DPL / 2; ++e) {
            v[2 * e] = __uint_as_float(raw.w[e] << 16);
            v[2 * e + 1] = __uint_as_float(raw.w[e] & 0xFFFF0000u);
          }
          static_for<G>([&](auto h) {
            // p for (key kbase+16t+4*row+j, head h) sits in lane (row, h), register j.
            const float ph = row_lane<h>(sc[t][j]);
#pragma unroll
            for (int d = 0; d < DPL; ++d) acc[h * DPL + d] = fmaf(ph, v[d], acc[h * DPL + d]);
          });
        }
      }
    };

    if constexpr (AHEAD) {
      TilePages following = {0, 0};
      if constexpr (ALIGNED && decltype(next)::value) following = unit_pages(u + NW);
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        if (ubase + 16 * t < uend)
          group(ubase + 16 * t, [&](int, int i) { return kr[t % PT][i]; }, [&](int, int j) { return vr[t % PT][j]; });
        if (t + PT < kTiles) {
          issue(t % PT, ubase + 16 * (t + PT), pages, t + PT);
        } else if constexpr (decltype(next)::value) {
          if (t + PT == kTiles) pages = following;
          issue(t % PT, ubase + NW * kUnit + 16 * (t + PT - kTiles), pages, t + PT - kTiles);
        }
      }
    } else {
      constexpr int kStep = 16 * TPG;
      for (int kbase = ONE_UNIT ? start + wave * kStep : ubase; kbase < uend; kbase += ONE_UNIT ? NW * kStep : kStep) {
        const uint16_t* krow[TPG];
#pragma unroll
        for (int t = 0; t < TPG; ++t) krow[t] = krow_of(kbase + 16 * t);
        group(kbase, [&](int t, int i) { return load_k(krow[t], i); },
              [&](int t, int j) { return load_v<D>(vrow_of(kbase + 16 * t, j)); });
      }
    }

    // Sum the four key quarters, each row keeping its quarter of the accumulators: rows r and
    // r ^ 2 first, then r and r ^ 1.
#pragma unroll
    for (int i = 0; i < FL / 2; ++i) {
      swap32(acc[i], acc[i + FL / 2]);
      acc[i] = acc[i] + acc[i + FL / 2];
    }
#pragma unroll
    for (int i = 0; i < QF; ++i) {
      swap16(acc[i], acc[i + QF]);
      acc[i] = acc[i] + acc[i + QF];
    }

    if constexpr (UNITS) {
      const int64_t nu = (int64_t)p.ns * p.units;  // units per request and head in the workspace
      const int64_t ui = (int64_t)s * p.units + unit0 + u;
      if (row == 0 && col < G) {
        const int64_t pi = ((int64_t)b * p.H + g * G + col) * nu + ui;
        p.mp[pi] = m_run;
        p.lp[pi] = l_run;
      }
#pragma unroll
      for (int i = 0; i < QF; ++i) {
        const int f = row * QF + i;
        p.ap[(((int64_t)b * p.H + g * G + f / DPL) * nu + ui) * D + col * DPL + f % DPL] = acc[i];
      }
    } else if constexpr (ONE_UNIT) {
      m_tot = m_run;
      l_tot = l_run;
#pragma unroll
      for (int i = 0; i < QF; ++i) a_tot[i] = acc[i];
    } else {
      // merge_state of the running state with the unit's, the factors computed once per head
      const float mn = fmaxf(m_tot, m_run);
      const float c_old = (m_tot == kNegInf) ? 0.0f : exp2_hw(m_tot - mn);
      const float c_new = (m_run == kNegInf) ? 0.0f : exp2_hw(m_run - mn);
      l_tot = fmaf(l_tot, c_old, l_run * c_new);
      m_tot = mn;
#pragma unroll
      for (int i = 0; i < QF; ++i) {
        const int h = (row * QF + i) / DPL;  // same for runs of DPL flats
        a_tot[i] = fmaf(a_tot[i], shfl_f32(c_old, h), acc[i] * shfl_f32(c_new, h));
      }
    }
  };

  const int nunit = (end - start + kUnit - 1) / kUnit;
  if constexpr (AHEAD) {
    if (wave < nunit) {
      if constexpr (ALIGNED) pages = unit_pages(wave);
#pragma unroll
      for (int t = 0; t < PT; ++t) issue(t, start + wave * kUnit + 16 * t, pages, t);
      int u = wave;
      for (; u + NW < nunit; u += NW) unit(u, std::true_type{});
      unit(u, std::false_type{});
    }
  } else if constexpr (ONE_UNIT) {
    unit(0, std::false_type{});
  } else {
    for (int u = wave; u < nunit; u += NW) unit(u, std::false_type{});
  }
  if constexpr (UNITS) return;

  if (row == 0 && col < G) {
    s_m[wave][col] = m_tot;
    s_l[wave][col] = l_tot;
  }
#pragma unroll
  for (int i = 0; i < QF; ++i) {
    const int f = row * QF + i;
    s_acc[wave][f / DPL][col * DPL + f % DPL] = a_tot[i];
  }
  __syncthreads();

  // Fixed-order merge of the waves, then either the final output (single-segment request)
  // or the segment partial.
  const int H = p.H;
  const int nsb = need;
  for (int idx = threadIdx.x; idx < G * D; idx += 64 * NW) {
    const int h = idx / D, d = idx % D;
    float m = kNegInf, l = 0.0f, a = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) merge_state(m, l, a, s_m[w][h], s_l[w][h], s_acc[w][h][d]);
    const int head = g * G + h;
    if (nsb == 1) {
      float mm = kNegInf, ll = 0.0f, aa = 0.0f;
      merge_state(mm, ll, aa, m, l, a);
      store_f32_as(p.out, p.out_dtype, (int64_t)b * p.sot + (int64_t)head * p.soh + d, aa / ll);
    } else {
      const int64_t pi = ((int64_t)b * H + head) * p.ns + s;
      if (d == 0) {
        p.mp[pi] = m;
        p.lp[pi] = l;
      }
      p.ap[pi * D + d] = a;
    }
  }
}

// Merge of the units of one (request, head), one workgroup of 16 waves, in the order of the
// whole-segment kernel: wave w's units of a segment (w, w + NW, ...), the NW waves, then the
// segments. A pass takes kSegs segments: their kSegs * NW unit chains go to groups of GL lanes (kBatch
// units loaded at once, so that a chain costs about one memory latency), the segments' waves are
// merged side by side, and one group appends the segments. What bounds a few long requests is the
// rate at which one CU loads (133 KB of partials per head at 16384 keys): SPLIT spreads a head's
// dims over D / 32 workgroups while that leaves at most one per CU. One request of 16384 keys, 32
// heads of 128: 5.8 -> 4.2 us; with 192 heads of 256 (12 requests) it would take 9.7 instead of 4.4.
template <int D, int NW, bool SPLIT>
__global__ __launch_bounds__(1024) void paged_merge_units_kernel(PagedParams p) {
  constexpr int GL = SPLIT ? 32 : 64;      // lanes of a group
  constexpr int DPL = SPLIT ? 1 : D / 64;  // dims of a lane
  constexpr int MD = GL * DPL;             // dims of the workgroup
  constexpr int kSegs = 8;
  constexpr int kBatch = 8;
  constexpr int kChains = kSegs * NW;
  constexpr int kGroups = 1024 / GL;
  __shared__ float c_m[kChains], c_l[kChains], c_a[kChains][MD];
  __shared__ float g_m[kSegs], g_l[kSegs], g_a[kSegs][MD];
  const int64_t bh = blockIdx.x / (D / MD);
  const int d0 = (int)(blockIdx.x % (D / MD)) * MD;
  const int b = (int)(bh / p.H);
  const int head = (int)(bh % p.H);
  if (p.n_live != nullptr && b >= *p.n_live) return;
  const int L = p.sl[b];
  const int nsb = min((L + p.split - 1) / p.split, p.ns_model);
  if (nsb > p.ns) return;  // NaN rows, written by the partial kernel
  if (nsb <= 0 && p.ns == 1) return;  // an empty request: as the whole-segment kernel leaves it
  const int lane = threadIdx.x % GL;
  const int group = threadIdx.x / GL;
  const int64_t base = bh * p.ns * p.units;
  float m = kNegInf, l = 0.0f, a = 0.0f;  // the request so far: thread d < MD holds its dim
  for (int s0 = 0; s0 < nsb; s0 += kSegs) {
    const int nseg = min(kSegs, nsb - s0);
    for (int c = group; c < nseg * NW; c += kGroups) {
      const int s = s0 + c / NW;
      const int keys = min(p.split, L - s * p.split);
      const int nunit = (keys + kUnit - 1) / kUnit;  // of the segment; this chain: c % NW, + NW, ...
      const int64_t u0 = base + (int64_t)s * p.units;
      float cm = kNegInf, cl = 0.0f, ca[DPL];
#pragma unroll
      for (int j = 0; j < DPL; ++j) ca[j] = 0.0f;
      for (int u = c % NW; u < nunit; u += NW * kBatch) {
        float ms[kBatch], ls[kBatch], as_[kBatch][DPL];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          // a unit past the segment's last repeats the first of the batch and is not merged
          const int64_t ui = u0 + (u + NW * k < nunit ? u + NW * k : u);
          ms[k] = p.mp[ui];
          ls[k] = p.lp[ui];
#pragma unroll
          for (int j = 0; j < DPL; ++j) as_[k][j] = p.ap[ui * D + d0 + lane + GL * j];
        }
        asm volatile("" ::: "memory");  // every load of the batch is issued before the first is used
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          if (u + NW * k >= nunit) break;
          const float m0 = cm, l0 = cl;
#pragma unroll
          for (int j = 0; j < DPL; ++j) {
            cm = m0;
            cl = l0;
            merge_state(cm, cl, ca[j], ms[k], ls[k], as_[k][j]);
          }
        }
      }
      if (lane == 0) {
        c_m[c] = cm;
        c_l[c] = cl;
      }
#pragma unroll
      for (int j = 0; j < DPL; ++j) c_a[c][lane + GL * j] = ca[j];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nseg * MD; i += 1024) {
      const int sg = i / MD, d = i % MD;
      float sm = kNegInf, sl = 0.0f, sa = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) merge_state(sm, sl, sa, c_m[sg * NW + w], c_l[sg * NW + w], c_a[sg * NW + w][d]);
      if (d == 0) {
        g_m[sg] = sm;
        g_l[sg] = sl;
      }
      g_a[sg][d] = sa;
    }
    __syncthreads();
    if (threadIdx.x < MD)
      for (int sg = 0; sg < nseg; ++sg) merge_state(m, l, a, g_m[sg], g_l[sg], g_a[sg][threadIdx.x]);
    // the next pass writes g_* only past its first barrier, and c_* were read before the last one
  }
  if (threadIdx.x < MD)
    store_f32_as(p.out, p.out_dtype, (int64_t)b * p.sot + (int64_t)head * p.soh + d0 + threadIdx.x, a / l);
}

template <int D>
void launch_merge_units(const PagedParams& pp, int64_t heads, hipStream_t st) {
  if (heads * (D / 32) <= 256)
    hipLaunchKernelGGL((paged_merge_units_kernel<D, 4, true>), dim3((unsigned)(heads * (D / 32))), dim3(1024), 0, st, pp);
  else
    hipLaunchKernelGGL((paged_merge_units_kernel<D, 4, false>), dim3((unsigned)heads), dim3(1024), 0, st, pp);
}

// Fixed-order merge over the segments of one (request, head); one wave per (b, head).
template <int D>
__global__ __launch_bounds__(64) void paged_merge_kernel(PagedParams p) {
  static_assert(D % 64 == 0, "a lane owns D / 64 columns");
  constexpr int DPW = D / 64;
  const int64_t bh = blockIdx.x;
  const int b = (int)(bh / p.H);
  const int head = (int)(bh % p.H);
  const int lane = threadIdx.x;
  // Segments are merged in index order, kChunk of them per pass, and a pass issues every load of
  // its segments first, so it waits for one memory latency rather than one per segment. The
  // first pass's loads go out before the request's length is read: they take segments
  // min(c, ns - 1), inside the workspace whatever the length; later passes clamp to the request's
  // last segment. A segment at or past that count is read and never merged.
  constexpr int kChunk = 8;
  const int64_t base = bh * p.ns;
  float ms[kChunk], ls[kChunk], as_[kChunk][DPW];
  auto load_pass = [&](int s0, int last) {
#pragma unroll
    for (int c = 0; c < kChunk; ++c) {
      const int64_t s = base + min(s0 + c, last);
      ms[c] = p.mp[s];
      ls[c] = p.lp[s];
#pragma unroll
      for (int j = 0; j < DPW; ++j) as_[c][j] = p.ap[s * D + lane + 64 * j];
    }
  };
  load_pass(0, p.ns - 1);
  asm volatile("" ::: "memory");  // the loads above stay above the reads of the length below
  if (p.n_live != nullptr && b >= *p.n_live) return;
  const int L = p.sl[b];
  const int nsb = min((L + p.split - 1) / p.split, p.ns_model);
  if (nsb == 1 || nsb > p.ns) return;  // written by the partial kernel (NaN rows past a trimmed grid)
  float m[DPW], l[DPW], a[DPW];
#pragma unroll
  for (int j = 0; j < DPW; ++j) {
    m[j] = kNegInf;
    l[j] = 0.0f;
    a[j] = 0.0f;
  }
  for (int s0 = 0;;) {
#pragma unroll
    for (int c = 0; c < kChunk; ++c) {
      if (s0 + c >= nsb) break;
#pragma unroll
      for (int j = 0; j < DPW; ++j) merge_state(m[j], l[j], a[j], ms[c], ls[c], as_[c][j]);
    }
    s0 += kChunk;
    if (s0 >= nsb) break;
    load_pass(s0, nsb - 1);
  }
#pragma unroll
  for (int j = 0; j < DPW; ++j) {
    const int d = lane + 64 * j;
    store_f32_as(p.out, p.out_dtype, (int64_t)b * p.sot + (int64_t)head * p.soh + d, a[j] / l[j]);
  }
}

// LDS bytes of a segment's block-table entries (the pages a `split`-key window can touch).
size_t page_table_bytes(int64_t split, int64_t bs) { return (size_t)(split / bs + 2) * sizeof(int32_t); }

enum PagedMode { kSegments = 0, kUnits = 1 };

template <int D, int G, int TPG, int NW, bool UNITS, bool AHEAD, bool ALIGNED>
hipError_t launch_partial(const PagedParams& pp, hipStream_t st) {
  const int64_t blocks = pp.n * pp.KV * pp.ns * (UNITS ? pp.slices : 1);
  if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  const int64_t keys = UNITS ? std::min<int64_t>(pp.split, pp.slice_units * kUnit) : pp.split;
  hipLaunchKernelGGL((paged_partial_kernel<D, G, TPG, NW, UNITS, AHEAD, ALIGNED>), dim3((unsigned)blocks), dim3(64 * NW),
                     page_table_bytes(keys, pp.bs), st, pp);
  return hipGetLastError();
}

template <int D, int G>
hipError_t dispatch_tpg_nw(int tpg, int nw, PagedMode mode, const PagedParams& pp, hipStream_t st) {
  // Pages of whole tiles, and lane offsets within a tile that fit 32 bits.
  const bool aligned = pp.bs % 16 == 0 && pp.skp >= 0 && pp.svp >= 0 && pp.skp < (1 << 25) && pp.svp < (1 << 25);
  if (nw == 4) {
    if (tpg == 1) {
      if (mode == kUnits)
        return aligned ? launch_partial<D, G, 1, 4, true, true, true>(pp, st)
                       : launch_partial<D, G, 1, 4, true, true, false>(pp, st);
      return aligned ? launch_partial<D, G, 1, 4, false, true, true>(pp, st)
                     : launch_partial<D, G, 1, 4, false, true, false>(pp, st);
    }
    if (tpg == 2) return launch_partial<D, G, 2, 4, false, false, false>(pp, st);
    if (tpg == 4) return launch_partial<D, G, 4, 4, false, false, false>(pp, st);
  } else if (nw == 8) {
    if (tpg == 1) return launch_partial<D, G, 1, 8, false, false, false>(pp, st);
    if (tpg == 2) return launch_partial<D, G, 2, 8, false, false, false>(pp, st);
    if (tpg == 4) return launch_partial<D, G, 4, 8, false, false, false>(pp, st);
  }
  return hipErrorInvalidValue;
}

template <int D>
hipError_t dispatch_g(int G, int tpg, int nw, PagedMode mode, const PagedParams& pp, hipStream_t st) {
  switch (G) {
    case 1: return dispatch_tpg_nw<D, 1>(tpg, nw, mode, pp, st);
    case 2: return dispatch_tpg_nw<D, 2>(tpg, nw, mode, pp, st);
    case 4: return dispatch_tpg_nw<D, 4>(tpg, nw, mode, pp, st);
    case 8: return dispatch_tpg_nw<D, 8>(tpg, nw, mode, pp, st);
    default: return hipErrorInvalidValue;
  }
}

int64_t num_segments(int64_t max_len, int64_t split) {
  const int64_t ns = (max_len + split - 1) / split;
  return ns < 1 ? 1 : ns;
}

int64_t units_of(int64_t split) { return cdiv<int64_t>(split, kUnit); }

size_t units_bytes(int64_t n, int64_t num_heads, int64_t head_dim, int64_t ns, int64_t split) {
  return (size_t)n * num_heads * ns * units_of(split) * (head_dim + 2) * sizeof(float);
}

// Whether the units of a grid of ns segments per request are computed apart. keys is the most
// keys a request of the grid may have. Measured at H32/KV8/D128 (us a call, whole segments /
// units): 1 request of 520 keys 13.1 / 10.9, 1024 18.5 / 11.2, 16384 35.3 / 21.2 (64 workgroups of
// whole segments); 2 of 16384 (128) 43.6 / 36.4; 4 of 16384 (256) 49.7 / 61.3; 16 of 1024 (128)
// 23.4 / 21.6; 32 of 1024 (256) 26.0 / 39.6. Past half the CUs the units' partials (an eighth of the
// keys' bytes, written and read back) cost more than the idle CUs. Up to 512 keys the merge launch
// costs what the shorter chains gain, unless a key is much work (G query heads of D dims): 1 request
// of 400 keys 8.9 / 9.1 at G = 4, D = 64, 11.7 / 10.8 at D = 128, 20.7 / 14.3 at D = 256, 9.1 / 9.5 at
// G = 1, D = 128, 17.6 / 13.1 at D = 256, 27.8 / 18.3 at G = 8, D = 256.
// The grid and the workspace hold every unit of a segment (a request past the caller's bound but inside
// its segment is computed too), so a segment much longer than the keys (more than 8 times their units)
// or partials past 256 MiB keep whole segments: 16 requests bounded by 1000 keys in segments of 131040
// would take 545 MB and 512 workgroups a head, 4 of them with keys. Segments of 2048 never do.
bool use_units(int64_t n, int64_t num_heads, int64_t kv_heads, int64_t head_dim, int64_t ns, int64_t split, int64_t keys,
               int64_t blk, int64_t waves) {
  const bool much = head_dim >= 256 || num_heads / kv_heads * head_dim >= 512;
  if (blk != 16 || waves != 4 || keys <= (much ? 4 : 8) * kUnit || n * kv_heads * ns > 128) return false;
  return units_of(split) <= 8 * units_of(keys) && units_bytes(n, num_heads, head_dim, ns, split) <= (size_t)256 << 20;
}

}  // namespace

extern "C" int vxa_paged_decode_units_workspace(int64_t n, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                                                int64_t max_len, int64_t split, int64_t blk, int64_t waves,
                                                size_t* ws_bytes) {
  const int rc = vxa_paged_decode_workspace(n, num_heads, head_dim, max_len, split, ws_bytes);
  if (rc != VXA_OK) return rc;
  if (num_kv_heads <= 0 || blk <= 0 || waves <= 0) return VXA_ERR_ARG;
  const int64_t ns = num_segments(max_len, split);
  if (use_units(n, num_heads, num_kv_heads, head_dim, ns, split, max_len, blk, waves))
    *ws_bytes = units_bytes(n, num_heads, head_dim, ns, split);
  return VXA_OK;
}

extern "C" int vxa_paged_decode_workspace(int64_t n, int64_t num_heads, int64_t head_dim, int64_t max_len,
                                          int64_t split, size_t* ws_bytes) {
  if (n < 0 || num_heads <= 0 || head_dim <= 0 || split <= 0 || !ws_bytes) return VXA_ERR_ARG;
  const int64_t ns = num_segments(max_len, split);
  *ws_bytes = ns > 1 ? (size_t)n * num_heads * ns * (head_dim + 2) * sizeof(float) : 0;
  return VXA_OK;
}

namespace {

int paged_decode_impl(const void* q, int64_t sqt, int64_t sqh, const void* k_cache, int64_t skb, int64_t skp,
                      int64_t skh, const void* v_cache, int64_t svb, int64_t svp, int64_t svh,
                      const int32_t* block_table, int64_t sbt, const int32_t* seq_lens, float scale, void* out,
                      int out_dtype, int64_t sot, int64_t soh, int64_t n, const int32_t* n_live,
                      int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, int64_t block_size,
                      int64_t max_len, int64_t max_seq_len, int64_t split, int64_t blk, int64_t waves, void* ws,
                      size_t ws_bytes, vxa_stream_t stream) {
  if (n < 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 || split <= 0 ||
      max_seq_len < 0)
    return VXA_ERR_ARG;
  if (out_dtype != VXA_F32 && out_dtype != VXA_BF16 && out_dtype != VXA_F16) return VXA_ERR_ARG;
  if (num_heads % num_kv_heads != 0) return VXA_ERR_ARG;
  if (n == 0) return VXA_OK;
  if (!q || !k_cache || !v_cache || !block_table || !seq_lens || !out) return VXA_ERR_ARG;
  const int64_t G = num_heads / num_kv_heads;
  if (split % 16 != 0 || split > (1 << 30)) return VXA_ERR_UNSUPPORTED;
  if (blk != 16 && blk != 32 && blk != 64) return VXA_ERR_UNSUPPORTED;
  if (waves != 4 && waves != 8) return VXA_ERR_UNSUPPORTED;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return VXA_ERR_UNSUPPORTED;
  if (G != 1 && G != 2 && G != 4 && G != 8) return VXA_ERR_UNSUPPORTED;
  if (block_size > (1 << 30) || num_heads > (1 << 20)) return VXA_ERR_UNSUPPORTED;
  if (page_table_bytes(split, block_size) > 32768) return VXA_ERR_UNSUPPORTED;  // split / block_size <= 8190
  // 16-byte row loads of q and V and 16/8-byte K fragments need aligned rows.
  if ((uintptr_t)q % 16 || (uintptr_t)k_cache % 16 || (uintptr_t)v_cache % 16 || sqt % 8 || sqh % 8 ||
      skb % 8 || skp % 8 || skh % 8 || svb % 8 || svp % 8 || svh % 8)
    return VXA_ERR_UNSUPPORTED;

  // The grid: the model's NS segments per request, or fewer when the caller bounds the batch's
  // lengths (max_seq_len > 0); the workspace holds the partials of the grid's segments.
  const int64_t ns_model = num_segments(max_len, split);
  const int64_t ns = max_seq_len > 0 ? std::min(ns_model, num_segments(max_seq_len, split)) : ns_model;
  size_t need = 0;
  vxa_paged_decode_workspace(n, num_heads, head_dim, ns * split, split, &need);
  if (need > 0 && (!ws || ws_bytes < need)) return VXA_ERR_WORKSPACE;

  PagedParams pp;
  pp.q = reinterpret_cast<const uint16_t*>(q);
  pp.sqt = sqt; pp.sqh = sqh;
  pp.kc = reinterpret_cast<const uint16_t*>(k_cache);
  pp.skb = skb; pp.skp = skp; pp.skh = skh;
  pp.vc = reinterpret_cast<const uint16_t*>(v_cache);
  pp.svb = svb; pp.svp = svp; pp.svh = svh;
  pp.bt = block_table; pp.sbt = sbt; pp.sl = seq_lens;
  pp.scale_log2 = (float)((double)scale * 1.4426950408889634);
  pp.split = (int32_t)split;
  pp.ns = (int32_t)ns;
  pp.ns_model = (int32_t)ns_model;
  pp.H = (int32_t)num_heads;
  pp.KV = (int32_t)num_kv_heads;
  pp.bs = (int32_t)block_size;
  pp.bs_shift = -1;
  if ((block_size & (block_size - 1)) == 0) {
    int sh = 0;
    while ((1LL << sh) < block_size) ++sh;
    pp.bs_shift = sh;
  }
  pp.n = n;
  pp.n_live = n_live;
  PagedMode mode = kSegments;
  const int64_t keys = max_seq_len > 0 ? std::min(max_len, max_seq_len) : max_len;
  if (use_units(n, num_heads, num_kv_heads, head_dim, ns, split, keys, blk, waves) && ws &&
      ws_bytes >= units_bytes(n, num_heads, head_dim, ns, split))
    mode = kUnits;
  pp.units = (int32_t)units_of(split);
  pp.slice_units = (int32_t)std::min<int64_t>(pp.units, waves);  // one unit per wave
  pp.slices = (int32_t)cdiv<int64_t>(pp.units, pp.slice_units);
  float* wsf = reinterpret_cast<float*>(ws);
  const int64_t nhs = n * num_heads * ns * (mode == kUnits ? pp.units : 1);
  const bool partials = ns > 1 || mode == kUnits;
  pp.mp = partials ? wsf : nullptr;
  pp.lp = partials ? wsf + nhs : nullptr;
  pp.ap = partials ? wsf + 2 * nhs : nullptr;
  pp.out = out; pp.sot = sot; pp.soh = soh; pp.out_dtype = out_dtype;

  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int tpg = (int)(blk / 16);
  const int nw = (int)waves;
  hipError_t err;
  switch (head_dim) {
    case 64: err = dispatch_g<64>((int)G, tpg, nw, mode, pp, st); break;
    case 128: err = dispatch_g<128>((int)G, tpg, nw, mode, pp, st); break;
    default: err = dispatch_g<256>((int)G, tpg, nw, mode, pp, st); break;
  }
  if (err == hipErrorInvalidValue) return VXA_ERR_UNSUPPORTED;
  if (err != hipSuccess) return VXA_ERR_LAUNCH;
  const int64_t blocks = n * num_heads;
  if (partials && blocks > 0x7FFFFFFFLL) return VXA_ERR_UNSUPPORTED;
  if (mode == kUnits) {
    switch (head_dim) {
      case 64: launch_merge_units<64>(pp, blocks, st); break;
      case 128: launch_merge_units<128>(pp, blocks, st); break;
      default: launch_merge_units<256>(pp, blocks, st); break;
    }
    if (hipGetLastError() != hipSuccess) return VXA_ERR_LAUNCH;
  } else if (ns > 1) {
    switch (head_dim) {
      case 64: hipLaunchKernelGGL(paged_merge_kernel<64>, dim3((unsigned)blocks), dim3(64), 0, st, pp); break;
      case 128: hipLaunchKernelGGL(paged_merge_kernel<128>, dim3((unsigned)blocks), dim3(64), 0, st, pp); break;
      default: hipLaunchKernelGGL(paged_merge_kernel<256>, dim3((unsigned)blocks), dim3(64), 0, st, pp); break;
    }
    if (hipGetLastError() != hipSuccess) return VXA_ERR_LAUNCH;
  }
  return VXA_OK;
}

}  // namespace

extern "C" int vxa_paged_decode(const void* q, int64_t sqt, int64_t sqh, const void* k_cache, int64_t skb,
                                int64_t skp, int64_t skh, const void* v_cache, int64_t svb, int64_t svp,
                                int64_t svh, const int32_t* block_table, int64_t sbt, const int32_t* seq_lens,
                                float scale, void* out, int out_dtype, int64_t sot, int64_t soh, int64_t n,
                                int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, int64_t block_size,
                                int64_t max_len, int64_t max_seq_len, int64_t split, int64_t blk, int64_t waves,
                                void* ws, size_t ws_bytes, vxa_stream_t stream) {
  return paged_decode_impl(q, sqt, sqh, k_cache, skb, skp, skh, v_cache, svb, svp, svh, block_table, sbt, seq_lens,
                           scale, out, out_dtype, sot, soh, n, nullptr, num_heads, num_kv_heads, head_dim,
                           block_size, max_len, max_seq_len, split, blk, waves, ws, ws_bytes, stream);
}

extern "C" int vxa_paged_decode_prefix(const void* q, int64_t sqt, int64_t sqh, const void* k_cache, int64_t skb,
                                       int64_t skp, int64_t skh, const void* v_cache, int64_t svb, int64_t svp,
                                       int64_t svh, const int32_t* block_table, int64_t sbt,
                                       const int32_t* seq_lens, float scale, void* out, int out_dtype,
                                       int64_t sot, int64_t soh, int64_t n, const int32_t* n_live,
                                       int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                                       int64_t block_size, int64_t max_len, int64_t max_seq_len, int64_t split,
                                       int64_t blk, int64_t waves, void* ws, size_t ws_bytes,
                                       vxa_stream_t stream) {
  if (n_live == nullptr) return VXA_ERR_ARG;
  return paged_decode_impl(q, sqt, sqh, k_cache, skb, skp, skh, v_cache, svb, svp, svh, block_table, sbt, seq_lens,
                           scale, out, out_dtype, sot, soh, n, n_live, num_heads, num_kv_heads, head_dim,
                           block_size, max_len, max_seq_len, split, blk, waves, ws, ws_bytes, stream);
}
