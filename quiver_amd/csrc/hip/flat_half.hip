// Flat exact search on the 16-bit matrix unit.
//
// The fp32 matrix instructions run at 157 TFLOP/s, the fp16 ones at 2.5 PFLOP/s with fp32
// accumulation. A float times a power of two splits into two halves, x = hi + lo with |lo| <= 2^-11
// |x|, and <q, x> = hi.hi + hi.lo + lo.hi up to 3 x 2^-22 of sum |q_i x_i|: three fp16 products give
// the dot product to about the rounding of an fp32 chain at a third of 16 times its rate. Where
// every stored value and every query of the batch is an integer of magnitude at most 2048, hi alone
// is exact and one product does.
//
// The scan does not keep rows but groups of 16 consecutive rows: a lane takes the minimum of its 16
// accumulators (one group of one query), and only that minimum is compared, queued and listed. The
// merge takes the best groups of a query, scores their rows in the reference's order and stops as
// soon as the rounding bound shows that no later group can hold a row of the answer. A result row is
// never decided by the 16-bit scan's value, only excluded by it, and every exclusion is covered by
// the bound (prep_queries_kernel) or the query goes to the exact kernel.
//
// Ranking value. Per query the scan ranks by s_q s_x (||x||^2 / 2 - <q, x>) (L2) or -s_q s_x <q, x>:
// the distance up to a positive factor and a constant of the query. s_x brings the largest stored
// norm to (2^10, 2^11], s_q the query's norm, both powers of two, so every half is in range. The
// norm enters as one more matrix step: three halves of ||x||^2 s_x^2 / 2^9 in the row's padding
// against (w, w, w), w = 2^8 s_q / s_x.
#include <type_traits>

#include "common.hpp"
#include "exact.hpp"
#include "flat_half.hpp"
#include "select.hpp"

namespace {

using namespace qvh;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = 8;  // 2 per SIMD: one's selection runs beside the other's matrix steps
constexpr int kThreads = kWaves * 64;
constexpr int kTile = static_cast<int>(kHalfTileRows);
// Queued groups per lane before a wave-wide flush (a 32-row block queues up to two). The queue arrays
// also carry the hand-off of two row waves: four query groups' lists, 4 * 64 * KL entries.
constexpr int queue_cap(int kl) { return kl > 16 ? 16 : 8; }
/// The three-product form with 64 queries per wave has no registers left for its lists: they live in
/// LDS, and a flush brings a lane's list into the accumulators' registers and back.
constexpr bool lists_in_lds(int np, int qg) { return np == 3 && qg == 2; }

/// Inserts (d, g) into the sorted list (the caller has checked d <= Ld[KL - 1]); a lane's groups come in
/// increasing order, so an equal minimum already listed stays ahead. One parallel step: every
/// entry's new value depends on its own compare and its neighbour's.
template <int KL>
__device__ __forceinline__ void group_insert(float (&Ld)[KL], uint32_t (&Lg)[KL], float d, uint32_t g) {
  bool lt[KL];
#pragma unroll
  for (int x = 0; x < KL; ++x) lt[x] = d < Ld[x];
#pragma unroll
  for (int x = KL - 1; x > 0; --x) {
    Ld[x] = lt[x] ? (lt[x - 1] ? Ld[x - 1] : d) : Ld[x];
    Lg[x] = lt[x] ? (lt[x - 1] ? Lg[x - 1] : g) : Lg[x];
  }
  Ld[0] = lt[0] ? d : Ld[0];
  Lg[0] = lt[0] ? g : Lg[0];
}

/// The same for groups in any order: equal minima by group.
template <int KL>
__device__ __forceinline__ void group_insert_any(float (&Ld)[KL], uint32_t (&Lg)[KL], float d, uint32_t g) {
  bool lt[KL];
#pragma unroll
  for (int x = 0; x < KL; ++x) lt[x] = (d < Ld[x]) | ((d == Ld[x]) & (g < Lg[x]));
#pragma unroll
  for (int x = KL - 1; x > 0; --x) {
    Ld[x] = lt[x] ? (lt[x - 1] ? Ld[x - 1] : d) : Ld[x];
    Lg[x] = lt[x] ? (lt[x - 1] ? Lg[x - 1] : g) : Lg[x];
  }
  Ld[0] = lt[0] ? d : Ld[0];
  Lg[0] = lt[0] ? g : Lg[0];
}

/// Minimum of 16 accumulators.
__device__ __forceinline__ float min16(const f32x16& a) {
  float m = fminf(fminf(a[0], a[1]), a[2]);
#pragma unroll
  for (int r = 3; r + 1 < 16; r += 2) m = fminf(fminf(m, a[r]), a[r + 1]);
  return fminf(m, a[15]);
}

// NK: 16-dim matrix steps per row. NP: 1 product (hi.hi) or 3. QG: 32-query column groups per wave.
// QG = 2: lane l lists query l of the wave's 64 (after one half-wave swap of the minima); QG = 1: the
// lanes j and j + 32 list the two 16-row halves of every block for query j of 32.
//
// Split of the work (1M x 128, 10,000 queries): 512 queries per work-group, so that a tile's
// conversion and LDS traffic is shared by as many queries as the registers hold (64 per wave: 128
// VGPRs of query halves at NP = 3), two waves per SIMD.
template <int NK, int KL, int NP, int QG>
__global__ void __launch_bounds__(kThreads) flat_half_kernel(HalfScanArgs a) {
  if (a.gate != nullptr && ((*a.gate != 0u) != (a.gate_want != 0u))) return;  // the same for the whole grid
  // A row in LDS: 16 NK halves, then 8 halves with the norm's three parts. The stride is 4 mod 8
  // banks, so 16 rows' 16-byte reads of one column touch every bank once.
  constexpr int STRIDE = 16 * NK + 8;
  constexpr int C8 = 2 * NK;  // 8-float chunks per row
  constexpr int CHUNKS = kTile * C8;
  constexpr int PER = (CHUNKS + kThreads - 1) / kThreads;
  __shared__ __attribute__((aligned(16))) _Float16 s_hi[2][kTile * STRIDE];
  __shared__ __attribute__((aligned(16))) _Float16 s_lo[NP == 3 ? 2 : 1][NP == 3 ? kTile * STRIDE : 8];
  __shared__ uint64_t s_bits[2];
  // Queued (minimum, group) per lane, entry-major.
  constexpr bool kLdsLists = lists_in_lds(NP, QG);
  constexpr int kCap = kLdsLists ? 4 : queue_cap(KL);
  __shared__ float s_qd[kCap * kThreads];
  __shared__ uint32_t s_qg[kCap * kThreads];
  __shared__ float s_ld[kLdsLists ? KL * kThreads : 1];  // entry-major
  __shared__ uint32_t s_lg[kLdsLists ? KL * kThreads : 1];
  static_assert(kLdsLists || 4 * 64 * KL <= kCap * kThreads, "the row waves' hand-off fits the queue arrays");

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;

  // Work-group w runs on XCD w % 8; each XCD gets its own row splits, so the work-groups resident on
  // one XCD at a time stream the same rows through its L2.
  uint32_t qb, split;
  const uint32_t wg = blockIdx.x;
  if (a.nsplit % 8 == 0) {
    const uint32_t x = wg % 8, li = wg / 8;
    split = (li / a.qblocks) * 8 + x;
    qb = li % a.qblocks;
  } else {
    split = wg / a.qblocks;
    qb = wg % a.qblocks;
  }

  const uint32_t rw = a.row_waves;
  const uint32_t qwaves = kWaves / rw;
  const uint32_t qgroup = static_cast<uint32_t>(wave) % qwaves;  // the wave's 32 QG queries
  const uint32_t rslot = static_cast<uint32_t>(wave) / qwaves;   // its 32-row half (rw = 2)
  const int blk0 = static_cast<int>(rslot), blk1 = rw == 1 ? 2 : blk0 + 1;
  const uint32_t q0 = (qb * qwaves + qgroup) * (32 * QG);
  const bool wave_active = q0 < a.nq;
  const uint32_t q = q0 + (QG == 2 ? static_cast<uint32_t>(lane) : static_cast<uint32_t>(j));  // the query this lane lists
  const bool qvalid = q < a.nq;
  const float sx = half_scale(stored_norm(a.meta, a.dp));

  // Query operands: column j of group g, dims 16 kk + 8 h .. + 7 of step kk, negated and scaled.
  f16x8 bh[QG][NK], bl[NP == 3 ? QG : 1][NP == 3 ? NK : 1];
  f16x8 baug[QG];
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    const uint32_t qc = q0 + 32 * g + j;
    const bool ok = qc < a.nq;
    const float sq = ok ? __uint_as_float(a.words[static_cast<size_t>(qc) * kHalfWordStride + kHalfScaleWord]) : 0.0f;
    const float* qp = a.Q + static_cast<size_t>(ok ? qc : 0) * a.dp;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const uint32_t c = static_cast<uint32_t>(16 * kk + 8 * h);
      const bool in = ok && c < a.dp;
      const f32x4 v0 = *reinterpret_cast<const f32x4*>(qp + (in ? c : 0));
      const f32x4 v1 = *reinterpret_cast<const f32x4*>(qp + (in ? c + 4 : 4));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float v = in ? -sq * (i < 4 ? v0[i & 3] : v1[i & 3]) : 0.0f;
        const _Float16 hi = static_cast<_Float16>(v);
        bh[g][kk][i] = hi;
        if constexpr (NP == 3) bl[g][kk][i] = static_cast<_Float16>(v - static_cast<float>(hi));
      }
    }
    const _Float16 w = static_cast<_Float16>(ok && h == 0 && a.l2 ? 256.0f * sq / sx : 0.0f);
    baug[g] = f16x8{w, w, w, 0, 0, 0, 0, 0};
  }

  // The lane's list, ascending; in LDS form only its last minimum stays in registers.
  constexpr int kRegs = kLdsLists ? 1 : KL;
  float Ld[kRegs];
  uint32_t Lg[kRegs];
#pragma unroll
  for (int x = 0; x < KL; ++x) {
    if constexpr (kLdsLists) {
      s_ld[x * kThreads + tid] = __builtin_huge_valf();
      s_lg[x * kThreads + tid] = QVH_EMPTY_ROW;
    } else {
      Ld[x] = __builtin_huge_valf();
      Lg[x] = QVH_EMPTY_ROW;
    }
  }
  float kth = __builtin_huge_valf();

  // Prune threshold: the smaller of this list's KL-th minimum and the shared per-query value. Any
  // list's KL-th bounds the KL-th of the union of all lists, so groups above it can never be among
  // the query's KL best (equal minima pass: ties are decided by group). A tighter shared bound from the
  // lists' best minima, one word per list, cost more in atomics than it pruned (50,000 x 64, k = 10,
  // scan and merge: 40 queries 115 us with it, 66 without; 256 queries 203 and 64; 1M x 128, 10,000
  // queries 3.18 ms a search and 3.05).
  uint32_t* const qw = a.words + static_cast<size_t>(qvalid ? q : 0u) * kHalfWordStride;
  float pthr = __builtin_huge_valf();
  if (qvalid && a.share) {
    pthr = ordered_to_float(__hip_atomic_load(qw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }
  constexpr uint32_t kLists = QG == 2 ? 1u : 2u;  // per split and query
  const uint32_t list = split * kLists + (QG == 2 ? 0u : static_cast<uint32_t>(h));
  auto share_threshold = [&]() {
    float t = kth;
    if constexpr (QG == 1) {
      // The lane pair's lists hold disjoint groups: their union has KL at or below
      // max(own[KL/2-1], other[KL/2-1]) as well as below either list's KL-th.
      const float oth_k = __shfl_xor(t, 32, 64);
      const float own_h = Ld[KL / 2 - 1], oth_h = __shfl_xor(own_h, 32, 64);
      t = fminf(fminf(t, oth_k), fmaxf(own_h, oth_h));
      if (a.share_rank != 0) {
        // The merge takes R > KL groups: the pair's union has 2 c >= R groups at or below the larger
        // of the two lanes' c-th entries.
        float own_c = Ld[0];
#pragma unroll
        for (int x = 1; x < KL; ++x) own_c = static_cast<uint32_t>(x) + 1 == a.share_rank ? Ld[x] : own_c;
        t = fmaxf(own_c, __shfl_xor(own_c, 32, 64));
      }
    }
    if (qvalid) {
      const uint32_t g = __hip_atomic_fetch_min(qw, float_to_ordered(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      t = fminf(t, ordered_to_float(g));
    }
    pthr = fminf(pthr, t);
  };

  int qcount = 0;
  float thr = pthr;
  auto flush_queue = [&]() {
    int m = qcount;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
    if (m == 0) return;
    auto insert_queued = [&](float(&D)[KL], uint32_t(&G)[KL]) {
      for (int e = 0; e < m; ++e) {
        if (e < qcount) {
          const float v = s_qd[e * kThreads + tid];
          if (v < D[KL - 1]) group_insert<KL>(D, G, v, s_qg[e * kThreads + tid]);
        }
      }
      kth = D[KL - 1];
    };
    if constexpr (kLdsLists) {
      float D[KL];
      uint32_t G[KL];
#pragma unroll
      for (int x = 0; x < KL; ++x) {
        D[x] = s_ld[x * kThreads + tid];
        G[x] = s_lg[x * kThreads + tid];
      }
      insert_queued(D, G);
#pragma unroll
      for (int x = 0; x < KL; ++x) {
        s_ld[x * kThreads + tid] = D[x];
        s_lg[x * kThreads + tid] = G[x];
      }
    } else {
      insert_queued(Ld, Lg);
    }
    qcount = 0;
    thr = fminf(pthr, kth);
  };

  const uint64_t r0 = static_cast<uint64_t>(split) * a.rows_per_split;
  const uint64_t r1 = r0 < a.n ? (a.n < r0 + a.rows_per_split ? a.n : r0 + a.rows_per_split) : r0;
  const uint32_t ntiles = static_cast<uint32_t>(ceil_div(r1 - r0, kTile));
  const uint64_t last_row = r1 > r0 ? r1 - 1 : r0;

  f32x4 stage[PER][2];
  float stage_norm = 0.0f;
  uint64_t stage_bits = ~0ull;
  // Unconditional loads (rows past the split repeat its last row, columns past the row its first:
  // masked later), so none sits under a branch and the next tile stays in flight under this one's
  // matrix steps.
  auto load_tile = [&](uint32_t t) {
    const uint64_t base = r0 + static_cast<uint64_t>(t) * kTile;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      int c = tid + p * kThreads;
      if (CHUNKS % kThreads != 0) c = c < CHUNKS ? c : CHUNKS - 1;
      const uint32_t row = static_cast<uint32_t>(c / C8), col = 8u * static_cast<uint32_t>(c % C8);
      uint64_t gr = base + row;
      gr = gr < last_row ? gr : last_row;
      const float* src_row = a.X + gr * a.dp + (col < a.dp ? col : 0u);
      stage[p][0] = *reinterpret_cast<const f32x4*>(src_row);
      stage[p][1] = *reinterpret_cast<const f32x4*>(src_row + 4);
    }
    if (a.l2) {
      uint64_t gn = base + (tid & (kTile - 1));
      gn = gn < last_row ? gn : last_row;
      stage_norm = a.xnorm[gn];
    }
    if (a.bitmap) stage_bits = a.bitmap[base >> 6];
  };
  // Row 16 h + 4 a + b of a 32-row block goes to LDS row 8 a + 4 h + b: accumulator register r of
  // lane half h is then row 16 h + r, so a lane's 16 accumulators are 16 consecutive rows.
  auto lds_row = [](uint32_t row) {
    return (row & 32u) | ((row >> 2 & 3u) << 3) | ((row >> 4 & 1u) << 2) | (row & 3u);
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int c = tid + p * kThreads;
      if (CHUNKS % kThreads == 0 || c < CHUNKS) {
        const uint32_t row = static_cast<uint32_t>(c / C8), col = 8u * static_cast<uint32_t>(c % C8);
        const float s = col < a.dp ? sx : 0.0f;
        f16x8 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float v = s * stage[p][i >> 2][i & 3];
          hi[i] = static_cast<_Float16>(v);
          if constexpr (NP == 3) lo[i] = static_cast<_Float16>(v - static_cast<float>(hi[i]));
        }
        const uint32_t at = lds_row(row) * STRIDE + col;
        *reinterpret_cast<f16x8*>(&s_hi[buf][at]) = hi;
        if constexpr (NP == 3) *reinterpret_cast<f16x8*>(&s_lo[buf][at]) = lo;
      }
    }
    if (tid < kTile) {
      float v = stage_norm * sx * sx * 0x1p-9f;
      f16x8 n = {};
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        n[i] = static_cast<_Float16>(v);
        v -= static_cast<float>(n[i]);
      }
      *reinterpret_cast<f16x8*>(&s_hi[buf][lds_row(static_cast<uint32_t>(tid)) * STRIDE + 16 * NK]) = n;
    }
    if (tid == kTile) s_bits[buf] = stage_bits;
  };

  if (ntiles > 0) {
    load_tile(0);
    store_tile(0);
    if (ntiles > 1) load_tile(1);
  }
  __syncthreads();

  // The next tile is converted into the other buffer in the middle of this one: its loads went out a
  // whole tile earlier, nothing waits for them next to the barrier, and the two waves of a SIMD
  // (w and w + 4) convert at different times, one's conversion beside the other's matrix steps.
  const int convert_at = wave < 4 ? 0 : 1;
  for (uint32_t t = 0; t < ntiles; ++t) {
    const int buf = static_cast<int>(t & 1);
    auto convert_next = [&]() {
      if (t + 1 < ntiles) {
        store_tile(buf ^ 1);
        if (t + 2 < ntiles) load_tile(t + 2);
      }
    };
    if (convert_at == 0 || !wave_active) convert_next();
    if (wave_active) {
      const uint64_t tile_row0 = r0 + static_cast<uint64_t>(t) * kTile;
      const uint64_t left = r1 - tile_row0;
      uint64_t admit = a.bitmap ? s_bits[buf] : ~0ull;
      if (left < 64) admit &= (1ull << left) - 1;
      admit = (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(admit >> 32)))) << 32) |
              static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(admit)));
      for (int blk = blk0; blk < blk1; ++blk) {
        const _Float16* ah = &s_hi[buf][(32 * blk + j) * STRIDE + 8 * h];
        // Every lane reads its row's norm parts; the upper half's weights are zero.
        const _Float16* an = &s_hi[buf][(32 * blk + j) * STRIDE + 16 * NK];
        auto frag = [](const _Float16* p) { return *reinterpret_cast<const f16x8*>(p); };
        f32x16 acc[QG];
#pragma unroll
        for (int g = 0; g < QG; ++g) acc[g] = f32x16{};
        // The LDS reads run ahead of the matrix steps that use them (a read takes longer than a
        // step's two or four matrix instructions); the scheduling barriers keep the compiler from
        // pulling each read down to its use. The norm step is last: without L2 its weights are zero.
        if constexpr (NP == 1) {
          f16x8 x[NK + 1];
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) x[kk] = frag(ah + 16 * kk);
          x[NK] = frag(an);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int kk = 0; kk <= NK; ++kk) {
#pragma unroll
            for (int g = 0; g < QG; ++g) {
              acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[kk], kk < NK ? bh[g][kk] : baug[g], acc[g], 0, 0, 0);
            }
          }
        } else {
          // The small products first: their roundings are 2^-11 of the sum's.
          const _Float16* al = &s_lo[buf][(32 * blk + j) * STRIDE + 8 * h];
          constexpr int AHEAD = 2;
          f16x8 xh[AHEAD + 1], xl[AHEAD + 1];
#pragma unroll
          for (int kk = 0; kk < AHEAD && kk < NK; ++kk) {
            xh[kk] = frag(ah + 16 * kk);
            xl[kk] = frag(al + 16 * kk);
          }
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) {
            if (kk + AHEAD < NK) {
              xh[(kk + AHEAD) % (AHEAD + 1)] = frag(ah + 16 * (kk + AHEAD));
              xl[(kk + AHEAD) % (AHEAD + 1)] = frag(al + 16 * (kk + AHEAD));
            }
            __builtin_amdgcn_sched_barrier(0);
            const f16x8 vh = xh[kk % (AHEAD + 1)], vl = xl[kk % (AHEAD + 1)];
#pragma unroll
            for (int g = 0; g < QG; ++g) acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, bh[g][kk], acc[g], 0, 0, 0);
#pragma unroll
            for (int g = 0; g < QG; ++g) acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, bl[g][kk], acc[g], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
          constexpr int AHEAD2 = 4;
          f16x8 x[AHEAD2 + 1];
          auto step = [&](int kk) { return frag(kk < NK ? ah + 16 * kk : an); };
#pragma unroll
          for (int kk = 0; kk < AHEAD2 && kk <= NK; ++kk) x[kk] = step(kk);
#pragma unroll
          for (int kk = 0; kk <= NK; ++kk) {
            if (kk + AHEAD2 <= NK) x[(kk + AHEAD2) % (AHEAD2 + 1)] = step(kk + AHEAD2);
            __builtin_amdgcn_sched_barrier(0);
            const f16x8 v = x[kk % (AHEAD2 + 1)];
#pragma unroll
            for (int g = 0; g < QG; ++g) {
              acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, kk < NK ? bh[g][kk] : baug[g], acc[g], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        const uint32_t bits = static_cast<uint32_t>(admit >> (32 * blk));
        if (bits != 0xFFFFFFFFu) {  // wave-uniform: a filter, or the split's last rows
          const uint32_t lb = bits >> (16 * h);
#pragma unroll
          for (int g = 0; g < QG; ++g) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[g][r] = (lb >> r) & 1u ? acc[g][r] : __builtin_huge_valf();
          }
        }
        const uint32_t group0 = static_cast<uint32_t>((tile_row0 + 32 * static_cast<uint32_t>(blk)) / kHalfGroupRows);
        if constexpr (QG == 2) {
          // Lane l gets the minima of both 16-row halves for query l of the wave's 64.
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(min16(acc[0])),
                                                           __float_as_uint(min16(acc[1])), false, false);
          const float m0 = __uint_as_float(sw[0]), m1 = __uint_as_float(sw[1]);
          // Groups at +inf (no admitted row) never pass; ties with the bound do. Lanes past the last
          // query never queue.
          const bool p0 = qvalid && m0 <= thr && m0 < __builtin_huge_valf();
          const bool p1 = qvalid && m1 <= thr && m1 < __builtin_huge_valf();
          if (__builtin_amdgcn_ballot_w64(p0 || p1)) {
            if (__builtin_amdgcn_ballot_w64(qcount > kCap - 2)) flush_queue();
            if (p0) {
              s_qd[qcount * kThreads + tid] = m0;
              s_qg[qcount * kThreads + tid] = group0;
              ++qcount;
            }
            if (p1) {
              s_qd[qcount * kThreads + tid] = m1;
              s_qg[qcount * kThreads + tid] = group0 + 1;
              ++qcount;
            }
          }
        } else {
          const float m = min16(acc[0]);
          const bool p = qvalid && m <= thr && m < __builtin_huge_valf();
          if (__builtin_amdgcn_ballot_w64(p)) {
            if (__builtin_amdgcn_ballot_w64(qcount > kCap - 1)) flush_queue();
            if (p) {
              s_qd[qcount * kThreads + tid] = m;
              s_qg[qcount * kThreads + tid] = group0 + static_cast<uint32_t>(h);
              ++qcount;
            }
          }
        }
        if (convert_at == 1 && blk == blk0) convert_next();
      }
      // Bounds are exchanged after tiles 0, 1, 3, 7 (the first rows move a bound the most), then every 8:
      // an exchange waits for a device-scope round trip (300,007 x 96, 1,003 queries, k = 30: every 64
      // tiles 0.88-0.99 ms a search, 32 0.95, 16 0.81, 8 0.72).
      if (t < 8 ? (t & (t + 1)) == 0 : t % 8 == 7) {
        flush_queue();
        if (a.share) {
          share_threshold();
          thr = fminf(pthr, kth);
        }
      }
    }
    __syncthreads();
  }

  if (wave_active) flush_queue();
  float D[KL];
  uint32_t G[KL];
#pragma unroll
  for (int x = 0; x < KL; ++x) {
    if constexpr (kLdsLists) {
      D[x] = s_ld[x * kThreads + tid];
      G[x] = s_lg[x * kThreads + tid];
    } else {
      D[x] = Ld[x];
      G[x] = Lg[x];
    }
  }
  if (rw == 2) {
    // The wave of the second halves (w + 4) hands its lists to the one of the first: through the
    // queue arrays, free once every wave has flushed, or where they are, in LDS.
    float* const hd = kLdsLists ? s_ld : s_qd;
    uint32_t* const hg = kLdsLists ? s_lg : s_qg;
    const uint32_t stride = kLdsLists ? kThreads : kThreads / 2;  // entry-major, 256 lanes hand over
    const uint32_t at = qgroup * 64 + static_cast<uint32_t>(lane) + (kLdsLists ? 256u : 0u);  // qgroup < 4
    __syncthreads();
    if (!kLdsLists && rslot == 1) {
#pragma unroll
      for (int x = 0; x < KL; ++x) {
        hd[x * stride + at] = D[x];
        hg[x * stride + at] = G[x];
      }
    }
    __syncthreads();
    if (rslot == 1) return;
    for (int x = 0; x < KL; ++x) {
      const float d = hd[x * stride + at];
      if (!__builtin_amdgcn_ballot_w64(d <= D[KL - 1] && d < __builtin_huge_valf())) break;
      group_insert_any<KL>(D, G, d, hg[x * stride + at]);
    }
  }
  if (qvalid) {
    // Back to distances: value / (s_q s_x), one power of two at a time.
    const float iq = 1.0f / __uint_as_float(qw[kHalfScaleWord]), ix = 1.0f / sx;
    const float qn = a.l2 ? a.qnorm[q] : 1.0f;
    const size_t o = (static_cast<size_t>(q) * (a.nsplit * kLists) + list) * KL;
#pragma unroll
    for (int x = 0; x < KL; ++x) {
      const float v = (a.l2 ? 2.0f : 1.0f) * (D[x] * iq * ix) + qn;
      a.part_d[o + x] = G[x] == QVH_EMPTY_ROW ? __builtin_huge_valf() : v;
      a.part_r[o + x] = G[x];
    }
  }
}

// ---- rows wider than 128 dims -----------------------------------------------------------------
//
// A 256-row x 256-query tile per work-group, accumulated over 32-dim chunks: wave w takes 128 rows
// (half w / 4) and 64 queries (w % 4) in 128 accumulators, so a 16-dim step reads 12 fragments from
// LDS for 24 matrix instructions (at 64 x 64 per wave the LDS, not the matrix unit, would be the
// limit). Rows are split into halves on their way into LDS; the queries come split, in fragment
// order, from a workspace written once per search, since their conversion would cost every
// work-group as much as the rows'. Selection happens once per tile and touches few values, so the
// lists live in the output arrays and only a lane with a passing group loads its own.
//
// Fragment (row block, step, half) in LDS: 64 slots of 16 bytes; lane (i, h) of the matrix step reads
// slot 32 h + (i ^ (4 h + 16 step)), a permutation that spreads the row loader's 8-byte stores over
// the banks.

constexpr int kWideTile = static_cast<int>(kHalfWideTileRows);

__global__ void __launch_bounds__(256) half_query_frags_kernel(const float* __restrict__ Q, uint32_t nq, uint32_t dp,
                                                               uint32_t steps, const uint32_t* __restrict__ words,
                                                               f16x8* __restrict__ out) {
  const uint64_t item = static_cast<uint64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);  // (query block, step)
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t qb = item / steps;
  const uint32_t step = static_cast<uint32_t>(item % steps);
  if (qb >= ceil_div(nq, 32)) return;
  const uint64_t q = qb * 32 + (lane & 31);
  const uint32_t c = step * 16 + 8 * (lane >> 5);
  const bool in = q < nq && c < dp;
  const float sq = in ? __uint_as_float(words[q * kHalfWordStride + kHalfScaleWord]) : 0.0f;
  const f32x4* src = reinterpret_cast<const f32x4*>(Q + (in ? q * dp + c : 0));
  const f32x4 v0 = src[0], v1 = src[1];
  f16x8 hi, lo;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float v = in ? -sq * (i < 4 ? v0[i & 3] : v1[i & 3]) : 0.0f;
    hi[i] = static_cast<_Float16>(v);
    lo[i] = static_cast<_Float16>(v - static_cast<float>(hi[i]));
  }
  out[item * 128 + lane] = hi;
  out[item * 128 + 64 + lane] = lo;
}

template <int KL>
__global__ void __launch_bounds__(kThreads) flat_half_wide_kernel(HalfScanArgs a) {
  constexpr int kFrag = 1024;                            // bytes
  constexpr int kXBytes = kWideTile / 32 * 2 * 2 * kFrag;  // 8 row blocks x 2 steps x (hi, lo)
  constexpr int kQBytes = static_cast<int>(kHalfWideQueries) / 32 * 2 * 2 * kFrag;
  __shared__ __attribute__((aligned(16))) unsigned char s_x[2][kXBytes];
  __shared__ __attribute__((aligned(16))) unsigned char s_q[2][kQBytes];
  __shared__ __attribute__((aligned(16))) f16x8 s_aug[2][kWideTile];  // the norm's three halves per row

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  uint32_t qb, split;
  const uint32_t wg = blockIdx.x;
  if (a.nsplit % 8 == 0) {  // XCD wg % 8 takes its own splits
    const uint32_t x = wg % 8, li = wg / 8;
    split = (li / a.qblocks) * 8 + x;
    qb = li % a.qblocks;
  } else {
    split = wg / a.qblocks;
    qb = wg % a.qblocks;
  }
  const int rhalf = wave >> 2;  // rows 128 rhalf .. + 127 of every tile
  const uint32_t q0 = qb * kHalfWideQueries + static_cast<uint32_t>(wave & 3) * 64;
  const bool wave_active = q0 < a.nq;
  const uint32_t q = q0 + static_cast<uint32_t>(lane);  // the query this lane lists
  const bool qvalid = q < a.nq;
  const float sx = half_scale(stored_norm(a.meta, a.dp));
  f16x8 baug[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const uint32_t qc = q0 + 32 * g + j;
    const float sq = qc < a.nq ? __uint_as_float(a.words[static_cast<size_t>(qc) * kHalfWordStride + kHalfScaleWord]) : 0.0f;
    const _Float16 w = static_cast<_Float16>(qc < a.nq && h == 0 && a.l2 ? 256.0f * sq / sx : 0.0f);
    baug[g] = f16x8{w, w, w, 0, 0, 0, 0, 0};
  }

  const uint32_t list = split * 2 + static_cast<uint32_t>(rhalf);
  uint32_t* const qw = a.words + static_cast<size_t>(qvalid ? q : 0u) * kHalfWordStride;
  float* const my_d = a.part_d + (static_cast<size_t>(qvalid ? q : 0u) * (2 * a.nsplit) + list) * KL;
  uint32_t* const my_g = a.part_r + (static_cast<size_t>(qvalid ? q : 0u) * (2 * a.nsplit) + list) * KL;
  if (qvalid) {
#pragma unroll
    for (int x = 0; x < KL; ++x) {
      my_d[x] = __builtin_huge_valf();
      my_g[x] = QVH_EMPTY_ROW;
    }
  }
  float kth = __builtin_huge_valf();
  float pthr = __builtin_huge_valf();

  const uint64_t r0 = static_cast<uint64_t>(split) * a.rows_per_split;
  const uint64_t r1 = r0 < a.n ? (a.n < r0 + a.rows_per_split ? a.n : r0 + a.rows_per_split) : r0;
  const uint32_t ntiles = static_cast<uint32_t>(ceil_div(r1 - r0, kWideTile));
  const uint32_t nchunks = (a.dp + 31) / 32;
  const uint32_t nsteps = ntiles * nchunks;
  const uint64_t last_row = r1 > r0 ? r1 - 1 : r0;
  const uint32_t qblocks32 = static_cast<uint32_t>(ceil_div(a.nq, 32));

  // Loader: 16 bytes (4 dims) of 4 rows per thread, a row's 8 pieces on adjacent lanes, and 64 bytes of
  // the query fragments. Unconditional loads at clamped addresses.
  f32x4 xs[4];
  f32x4 qs[4];
  float norm = 0.0f;
  const uint32_t col = static_cast<uint32_t>(tid & 7), row0 = static_cast<uint32_t>(tid >> 3);
  auto load_step = [&](uint32_t t, uint32_t c) {
    const uint64_t base = r0 + static_cast<uint64_t>(t) * kWideTile;
    const uint32_t d = c * 32 + col * 4;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      uint64_t gr = base + row0 + 64 * p;
      gr = gr < last_row ? gr : last_row;
      xs[p] = *reinterpret_cast<const f32x4*>(a.X + gr * a.dp + (d < a.dp ? d : 0u));
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const uint32_t unit = static_cast<uint32_t>(tid + p * kThreads);  // 256 units per 32 queries
      uint32_t b = qb * (kHalfWideQueries / 32) + unit / 256;
      b = b < qblocks32 ? b : qblocks32 - 1;
      qs[p] = reinterpret_cast<const f32x4*>(a.qfrag)[(static_cast<size_t>(b) * (2 * nchunks) + 2 * c) * 128 + unit % 256];
    }
    if (c == 0 && a.l2) {
      uint64_t gn = base + static_cast<uint32_t>(tid & (kWideTile - 1));
      gn = gn < last_row ? gn : last_row;
      norm = a.xnorm[gn];
    }
  };
  auto store_step = [&](uint32_t t, uint32_t c, int buf) {
    const uint32_t step = col >> 2, hh = (col >> 1) & 1u;
    const float s = c * 32 + col * 4 < a.dp ? sx : 0.0f;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const uint32_t row = row0 + 64 * p, i = (row >> 2 & 3u) << 3 | (row >> 4 & 1u) << 2 | (row & 3u);
      typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
      f16x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = s * xs[p][e];
        hi[e] = static_cast<_Float16>(v);
        lo[e] = static_cast<_Float16>(v - static_cast<float>(hi[e]));
      }
      const uint32_t at = ((row >> 5) * 2 + step) * 2 * kFrag + (32 * hh + (i ^ (4 * hh + 16 * step))) * 16 + (col & 1u) * 8;
      *reinterpret_cast<f16x4*>(&s_x[buf][at]) = hi;
      *reinterpret_cast<f16x4*>(&s_x[buf][at + kFrag]) = lo;
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) *reinterpret_cast<f32x4*>(&s_q[buf][(tid + p * kThreads) * 16]) = qs[p];
    if (c == 0 && tid < kWideTile) {
      float v = norm * sx * sx * 0x1p-9f;
      f16x8 n = {};
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        n[e] = static_cast<_Float16>(v);
        v -= static_cast<float>(n[e]);
      }
      const uint32_t row = static_cast<uint32_t>(tid);
      s_aug[t & 1][(row & ~31u) | (row >> 2 & 3u) << 3 | (row >> 4 & 1u) << 2 | (row & 3u)] = n;
    }
  };

  auto after = [&](uint32_t& tt, uint32_t& cc) {  // the step after (tt, cc)
    if (++cc == nchunks) {
      cc = 0;
      ++tt;
    }
  };
  if (nsteps > 0) {
    load_step(0, 0);
    store_step(0, 0, 0);
    uint32_t t1 = 0, c1 = 0;
    after(t1, c1);
    if (nsteps > 1) load_step(t1, c1);
  }
  __syncthreads();

  f32x16 acc[4][2];
  uint32_t t = 0, c = 0;
  for (uint32_t i = 0; i < nsteps; ++i) {
    const int buf = static_cast<int>(i & 1);
    uint32_t nt = t, nc = c;
    after(nt, nc);
    // As in the narrow scan: the next step goes into the other buffer from loads issued a step
    // earlier, the two waves of a SIMD at different times.
    auto convert_next = [&]() {
      if (i + 1 < nsteps) {
        store_step(nt, nc, buf ^ 1);
        uint32_t t2 = nt, c2 = nc;
        after(t2, c2);
        if (i + 2 < nsteps) load_step(t2, c2);
      }
    };
    if (wave < 4 || !wave_active) convert_next();
    if (wave_active) {
      if (c == 0) {
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          acc[rb][0] = f32x16{};
          acc[rb][1] = f32x16{};
        }
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const unsigned char* qbase = &s_q[buf][((2 * (wave & 3)) * 2 + kk) * 2 * kFrag + lane * 16];
        const f16x8 bh0 = *reinterpret_cast<const f16x8*>(qbase), bl0 = *reinterpret_cast<const f16x8*>(qbase + kFrag);
        const f16x8 bh1 = *reinterpret_cast<const f16x8*>(qbase + 4 * kFrag);
        const f16x8 bl1 = *reinterpret_cast<const f16x8*>(qbase + 5 * kFrag);
        const unsigned char* xbase = &s_x[buf][(4 * rhalf * 2 + kk) * 2 * kFrag + (32 * h + (j ^ (4 * h + 16 * kk))) * 16];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          const f16x8 ah = *reinterpret_cast<const f16x8*>(xbase + rb * 4 * kFrag);
          const f16x8 al = *reinterpret_cast<const f16x8*>(xbase + rb * 4 * kFrag + kFrag);
          acc[rb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh0, acc[rb][0], 0, 0, 0);
          acc[rb][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh1, acc[rb][1], 0, 0, 0);
          acc[rb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl0, acc[rb][0], 0, 0, 0);
          acc[rb][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl1, acc[rb][1], 0, 0, 0);
          acc[rb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh0, acc[rb][0], 0, 0, 0);
          acc[rb][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh1, acc[rb][1], 0, 0, 0);
        }
        if (kk == 0 && wave >= 4) convert_next();
      }
      if (c + 1 == nchunks) {
        const uint64_t wave_row0 = r0 + static_cast<uint64_t>(t) * kWideTile + 128 * static_cast<uint64_t>(rhalf);
        float m[8];  // the minima of this lane's query over the wave's eight 16-row groups
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          if (a.l2) {
            const f16x8 xn = s_aug[t & 1][128 * rhalf + 32 * rb + j];
            acc[rb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xn, baug[0], acc[rb][0], 0, 0, 0);
            acc[rb][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xn, baug[1], acc[rb][1], 0, 0, 0);
          }
          const uint64_t block0 = wave_row0 + 32 * static_cast<uint64_t>(rb);
          uint32_t bits = block0 >= r1 ? 0u : r1 - block0 < 32 ? (1u << (r1 - block0)) - 1u : 0xFFFFFFFFu;
          if (a.bitmap && bits) bits &= static_cast<uint32_t>(a.bitmap[block0 >> 6] >> (block0 & 32));
          bits = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(bits)));
          if (bits != 0xFFFFFFFFu) {
            const uint32_t lb = bits >> (16 * h);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              acc[rb][0][r] = (lb >> r) & 1u ? acc[rb][0][r] : __builtin_huge_valf();
              acc[rb][1][r] = (lb >> r) & 1u ? acc[rb][1][r] : __builtin_huge_valf();
            }
          }
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(min16(acc[rb][0])),
                                                           __float_as_uint(min16(acc[rb][1])), false, false);
          m[2 * rb] = __uint_as_float(sw[0]);
          m[2 * rb + 1] = __uint_as_float(sw[1]);
        }
        const float thr = fminf(pthr, kth);
        bool any = false;
#pragma unroll
        for (int e = 0; e < 8; ++e) any = any || (m[e] <= thr && m[e] < __builtin_huge_valf());
        if (qvalid && any) {
          float Ld[KL];
          uint32_t Lg[KL];
#pragma unroll
          for (int x = 0; x < KL; ++x) {
            Ld[x] = my_d[x];
            Lg[x] = my_g[x];
          }
          const uint32_t group0 = static_cast<uint32_t>(wave_row0 / kHalfGroupRows);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            if (m[e] <= thr && m[e] < Ld[KL - 1]) group_insert<KL>(Ld, Lg, m[e], group0 + e);
          }
#pragma unroll
          for (int x = 0; x < KL; ++x) {
            my_d[x] = Ld[x];
            my_g[x] = Lg[x];
          }
          kth = Ld[KL - 1];
        }
        // The shared bound, as in the narrow scan; a tile is long enough to exchange it after each. Where
        // the merge takes more than KL groups (share is 0) only this list's own bound prunes.
        if (a.share && qvalid) {
          const uint32_t g = __hip_atomic_fetch_min(qw, float_to_ordered(kth), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          pthr = fminf(pthr, fminf(kth, ordered_to_float(g)));
        }
      }
    }
    t = nt;
    c = nc;
    __syncthreads();
  }

  if (qvalid) {
    const float iq = 1.0f / __uint_as_float(qw[kHalfScaleWord]), ix = 1.0f / sx;
    const float qn = a.l2 ? a.qnorm[q] : 1.0f;
#pragma unroll
    for (int x = 0; x < KL; ++x) {
      if (my_g[x] != QVH_EMPTY_ROW) my_d[x] = (a.l2 ? 2.0f : 1.0f) * (my_d[x] * iq * ix) + qn;
    }
  }
}

// ---- merge: the best groups, scored exactly ---------------------------------------------------

constexpr int kHeld = 4;  // keys held per list before it reloads

/// Keys p .. p + kHeld - 1 of one list (positions at or past KL read the list's start, never used).
template <int KL>
__device__ __forceinline__ void load_held(const float* ld, const uint32_t* lg, uint32_t p, float (&d)[kHeld],
                                          uint32_t (&g)[kHeld]) {
  static_assert(kHeld == 4, "one 16-byte load per list");
  if constexpr (KL % 4 == 0) {
    const uint32_t at = p + 4 <= KL ? p : 0u;
    const f32x4 dv = *reinterpret_cast<const f32x4*>(ld + at);
    const f32x4 gv = *reinterpret_cast<const f32x4*>(lg + at);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      d[i] = dv[i];
      g[i] = __float_as_uint(gv[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t at = p + i < KL ? p + i : 0u;
      d[i] = ld[at];
      g[i] = lg[at];
    }
  }
}

/// The m.sel best groups over a query's lists, ascending by (minimum, group), into sel: popped by one
/// wave from list heads held in registers (LPL lists per lane). Returns their count; *spent: some list
/// gave all of its entries before the selection ended.
template <int KL, int LPL>
__device__ __forceinline__ uint32_t select_groups(const HalfMergeArgs& m, uint32_t q, uint64_t* sel, bool* spent) {
  const int lane = threadIdx.x & 63;
  const float* pd = m.part_d + static_cast<size_t>(q) * m.nlists * KL;
  const uint32_t* pg = m.part_r + static_cast<size_t>(q) * m.nlists * KL;
  uint64_t kk[LPL][kHeld];
  uint32_t ptr[LPL];
#pragma unroll
  for (int u = 0; u < LPL; ++u) {
    ptr[u] = 0;
    if (64u * u < m.nlists) {  // wave-uniform
      const uint32_t li = lane + 64 * u;
      const bool ok = li < m.nlists;
      const uint32_t lc = ok ? li : 0u;
      float d[kHeld];
      uint32_t g[kHeld];
      load_held<KL>(pd + static_cast<size_t>(lc) * KL, pg + static_cast<size_t>(lc) * KL, 0, d, g);
#pragma unroll
      for (int i = 0; i < kHeld; ++i) kk[u][i] = ok && i < KL ? make_key(d[i], g[i]) : ~0ull;
    } else {
#pragma unroll
      for (int i = 0; i < kHeld; ++i) kk[u][i] = ~0ull;
    }
  }
  uint32_t count = 0;
  bool out = false;
  for (uint32_t x = 0; x < m.sel; ++x) {
    uint64_t mine = kk[0][0];
    int arg = 0;
#pragma unroll
    for (int u = 1; u < LPL; ++u) {
      if (kk[u][0] < mine) {
        mine = kk[u][0];
        arg = u;
      }
    }
    const uint64_t best = wave_min_u64(mine);
    if (static_cast<uint32_t>(best) == QVH_EMPTY_ROW) break;  // only empty slots remain
    if (lane == 0) sel[x] = best;
    ++count;
    if (mine == best) {
#pragma unroll
      for (int u = 0; u < LPL; ++u) {
        if (u == arg) {
#pragma unroll
          for (int i = 0; i + 1 < kHeld; ++i) kk[u][i] = kk[u][i + 1];
          kk[u][kHeld - 1] = ~0ull;
          const uint32_t p = ++ptr[u];
          if (p == KL) out = out || x + 1 < m.sel;
          if (p % kHeld == 0 && p < KL) {
            float d[kHeld];
            uint32_t g[kHeld];
            load_held<KL>(pd + static_cast<size_t>(lane + 64 * u) * KL, pg + static_cast<size_t>(lane + 64 * u) * KL, p,
                          d, g);
#pragma unroll
            for (int i = 0; i < kHeld; ++i) kk[u][i] = p + i < KL ? make_key(d[i], g[i]) : ~0ull;
          }
        }
      }
    }
  }
  *spent = __ballot(out) != 0;
  return count;
}

/// One wave scores the 64 rows of groups sel[c0 .. c0 + 3] (below count) in the reference's order, eight
/// lanes per row, and returns their (distance, row) keys sorted, one per lane (absent rows last).
__device__ __forceinline__ uint64_t score_groups(const HalfMergeArgs& m, const float* qp, const uint64_t* sel,
                                                 uint32_t c0, uint32_t count, uint64_t* keys) {
  const int lane = threadIdx.x & 63;
  const uint32_t oct = static_cast<uint32_t>(lane) >> 3;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const float* b[4];
    uint32_t row[4];
    bool ok[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t e = static_cast<uint32_t>(pass) * 32 + static_cast<uint32_t>(c) * 8 + oct;  // row of the 64
      const uint32_t gi = c0 + e / 16;
      ok[c] = gi < count;
      const uint64_t pos = static_cast<uint64_t>(static_cast<uint32_t>(sel[ok[c] ? gi : 0])) * kHalfGroupRows + e % 16;
      ok[c] = ok[c] && pos < m.n;
      row[c] = ok[c] ? (m.idx ? m.idx[pos] : static_cast<uint32_t>(pos)) : 0u;
      if (m.bitmap) ok[c] = ok[c] && ((m.bitmap[row[c] >> 6] >> (row[c] & 63)) & 1u);
      b[c] = ok[c] ? m.X + static_cast<size_t>(row[c]) * m.dp : qp;
    }
    float e4[4];
    if (m.l2) {
      exact_group8_lines<true, 4>(qp, b, m.dim, e4);
    } else {
      exact_group8_lines<false, 4>(qp, b, m.dim, e4);
    }
    if ((lane & 7) == 0) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float d = m.l2 ? e4[c] : 1.0f - e4[c];
        d = d == d ? d : __builtin_huge_valf();
        keys[pass * 32 + c * 8 + static_cast<int>(oct)] = ok[c] ? make_key(d, row[c]) : ~0ull;
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
  uint64_t key[1] = {keys[lane]};
  wave_sort<1>(key);
  __builtin_amdgcn_wave_barrier();
  return key[0];
}

/// The 64 smallest of two sorted lists of 64 keys, one per lane: `best` and, reversed, `other`.
__device__ __forceinline__ uint64_t merge64(uint64_t best, uint64_t other_reversed) {
  uint64_t v[1] = {best < other_reversed ? best : other_reversed};
  wave_merge<1>(v);
  return v[0];
}

/// First the `sel` best groups over the query's lists. Then their rows in the reference's order, keeping
/// the best (distance, row), 64 rows per wave and step. After each step the next group's minimum
/// decides: every row not yet scored has a scan distance of at least that, so an exact one of at least
/// that minus delta, and once this is above the k-th best distance the answer is final. At the end
/// of the selection the answer stands if the lists held no more groups or if delta is 0 (the scan's
/// distances are exact: the sel >= k selected minima are rows that precede every row of any other
/// group in (distance, row) order); otherwise the last selected minimum decides the same way, and a
/// query that fails goes to the exact kernel.
///
/// W = 1: one wave per query, four queries per work-group. In a large batch the reads of the scored
/// rows bound it (10,000 queries of 12 groups x 16 rows x 512 bytes), and it stops after the fewest.
/// W = 4: four waves per query score 16 groups per step, for batches too small to fill the chip, where
/// the chain of dependent reads counts. LPL = 1 where a query has at most 64 lists: the eight lists
/// per lane of the other form cost registers that hold a third of the waves.
template <int KL, int LPL, int W>
__global__ void __launch_bounds__(256) flat_half_merge_kernel(HalfMergeArgs m) {
  if (m.gate != nullptr && ((*m.gate != 0u) != (m.gate_want != 0u))) return;
  __shared__ uint64_t s_sel[4][kHalfMaxSel];
  __shared__ uint64_t s_key[4][64];
  __shared__ uint32_t s_state[2];  // W = 4: count (or ~0 when the query falls back), done
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t q = W == 4 ? blockIdx.x : blockIdx.x * 4 + wave;
  if (q >= m.nq) return;  // W = 1: whole waves, no block barriers; W = 4: never
  uint64_t* const sel = s_sel[W == 4 ? 0 : wave];
  const double delta = static_cast<double>(m.delta[q]);
  const bool lead = W == 1 || wave == 0;
  uint32_t count = 0;
  bool failed = false;
  if (lead) {
    bool spent = false;
    count = select_groups<KL, LPL>(m, q, sel, &spent);
    // A list that ran out (wide merge) may have held more of the answer; a non-finite bound certifies
    // nothing.
    failed = (m.wide && spent) || !(delta < static_cast<double>(__builtin_huge_valf()));
  }
  if constexpr (W == 4) {
    if (threadIdx.x == 0) s_state[0] = failed ? ~0u : count;
    __syncthreads();
    count = s_state[0];
    failed = count == ~0u;
  } else {
    __builtin_amdgcn_wave_barrier();
  }
  if (failed) {
    if (lead && lane == 0) m.fallback[atomicAdd(m.nfallback, 1u)] = q;
    return;
  }

  const float* qp = m.Q + static_cast<size_t>(q) * m.dp;
  const uint32_t k = m.k;  // at most 64
  uint64_t best = ~0ull;   // the 64 best keys so far, ascending over the lanes (the leading wave's)
  uint64_t kth = ~0ull;
  bool done = false;
  for (uint32_t c0 = 0; c0 < count && !done; c0 += 4 * W) {
    const uint64_t mine = score_groups(m, qp, sel, c0 + (W == 4 ? 4u * static_cast<uint32_t>(wave) : 0u), count, s_key[wave]);
    s_key[wave][lane] = mine;
    if constexpr (W == 4) {
      __syncthreads();
      if (wave == 0) {
#pragma unroll
        for (int w = 0; w < 4; ++w) best = merge64(best, s_key[w][63 - lane]);
      }
    } else {
      __builtin_amdgcn_wave_barrier();
      best = merge64(best, s_key[wave][63 - lane]);
      __builtin_amdgcn_wave_barrier();
    }
    if (lead) {
      kth = __shfl(best, static_cast<int>(k) - 1, 64);
      if (kth != ~0ull && c0 + 4 * W < count) {
        const double g_next = static_cast<double>(ordered_to_float(static_cast<uint32_t>(sel[c0 + 4 * W] >> 32)));
        done = g_next - delta > static_cast<double>(ordered_to_float(static_cast<uint32_t>(kth >> 32)));
      }
    }
    if constexpr (W == 4) {
      if (threadIdx.x == 0) s_state[1] = done ? 1u : 0u;
      __syncthreads();
      done = s_state[1] != 0u;
    }
  }
  if (!lead) return;
  if (!done && count >= m.sel && delta != 0.0) {
    const double g_last = static_cast<double>(ordered_to_float(static_cast<uint32_t>(sel[count - 1] >> 32)));
    const bool certified =
        kth != ~0ull && static_cast<double>(ordered_to_float(static_cast<uint32_t>(kth >> 32))) < g_last - delta;
    if (!certified) {
      if (lane == 0) m.fallback[atomicAdd(m.nfallback, 1u)] = q;
      return;
    }
  }
  if (static_cast<uint32_t>(lane) < k) {
    const bool full = best != ~0ull;
    m.out_rows[static_cast<size_t>(q) * k + lane] = full ? static_cast<uint32_t>(best) : QVH_EMPTY_ROW;
    m.out_dist[static_cast<size_t>(q) * k + lane] =
        full ? ordered_to_float(static_cast<uint32_t>(best >> 32)) : __builtin_huge_valf();
  }
}

template <int KL>
void launch_merge_kl(const HalfMergeArgs& m, hipStream_t s) {
  const bool four = m.nq <= kHalfMergeFour;
  const dim3 grid(static_cast<unsigned>(four ? m.nq : ceil_div(m.nq, 4)));
  auto kernel = m.nlists <= 64 ? (four ? flat_half_merge_kernel<KL, 1, 4> : flat_half_merge_kernel<KL, 1, 1>)
                               : (four ? flat_half_merge_kernel<KL, 8, 4> : flat_half_merge_kernel<KL, 8, 1>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, m);
}

template <int NK>
void launch_nk(int kl, int products, bool pair, dim3 grid, const HalfScanArgs& a, hipStream_t s) {
  if (products == 1) {
    if (kl != 10) throw Failure(QVH_EUNSUPPORTED, "half scan: one product takes lists of 10");
    if (pair) {
      hipLaunchKernelGGL((flat_half_kernel<NK, 10, 1, 1>), grid, dim3(kThreads), 0, s, a);
    } else {
      hipLaunchKernelGGL((flat_half_kernel<NK, 10, 1, 2>), grid, dim3(kThreads), 0, s, a);
    }
  } else if (kl == 16) {
    if (pair) {
      hipLaunchKernelGGL((flat_half_kernel<NK, 16, 3, 1>), grid, dim3(kThreads), 0, s, a);
    } else {
      hipLaunchKernelGGL((flat_half_kernel<NK, 16, 3, 2>), grid, dim3(kThreads), 0, s, a);
    }
  } else if (kl == 32 && pair) {
    hipLaunchKernelGGL((flat_half_kernel<NK, 32, 3, 1>), grid, dim3(kThreads), 0, s, a);
  } else {
    throw Failure(QVH_EUNSUPPORTED, "half scan: unsupported list length");
  }
}

}  // namespace

namespace qvh {

void launch_half_scan(int kl, int products, bool pair, dim3 grid, const HalfScanArgs& a, hipStream_t s) {
  switch ((a.dp + 15) / 16) {
    case 1: launch_nk<1>(kl, products, pair, grid, a, s); break;
    case 2: launch_nk<2>(kl, products, pair, grid, a, s); break;
    case 3: launch_nk<3>(kl, products, pair, grid, a, s); break;
    case 4: launch_nk<4>(kl, products, pair, grid, a, s); break;
    case 5: launch_nk<5>(kl, products, pair, grid, a, s); break;
    case 6: launch_nk<6>(kl, products, pair, grid, a, s); break;
    case 7: launch_nk<7>(kl, products, pair, grid, a, s); break;
    case 8: launch_nk<8>(kl, products, pair, grid, a, s); break;
    default: throw Failure(QVH_EUNSUPPORTED, "half scan: unsupported row width");
  }
}

void launch_half_query_frags(const float* Q, uint32_t nq, uint32_t dp, const uint32_t* words, void* out,
                             hipStream_t s) {
  const uint64_t steps = half_wide_steps(dp), items = ceil_div(nq, 32) * steps;
  hipLaunchKernelGGL(half_query_frags_kernel, dim3(static_cast<unsigned>(ceil_div(items, 4))), dim3(256), 0, s, Q, nq,
                     dp, static_cast<uint32_t>(steps), words, static_cast<f16x8*>(out));
}

void launch_half_wide_scan(int kl, dim3 grid, const HalfScanArgs& a, hipStream_t s) {
  if (a.gate != nullptr) throw Failure(QVH_EUNSUPPORTED, "half scan: the wide form takes no gate");
  if (kl == 16) {
    hipLaunchKernelGGL(flat_half_wide_kernel<16>, grid, dim3(kThreads), 0, s, a);
  } else {
    hipLaunchKernelGGL(flat_half_wide_kernel<32>, grid, dim3(kThreads), 0, s, a);
  }
}

void launch_half_merge(int kl, const HalfMergeArgs& m, hipStream_t s) {
  static_assert(kHalfMaxLists <= 8 * 64, "eight lists per lane");
  if (kl == 10) {
    launch_merge_kl<10>(m, s);
  } else if (kl == 16) {
    launch_merge_kl<16>(m, s);
  } else {
    launch_merge_kl<32>(m, s);
  }
}

}  // namespace qvh
