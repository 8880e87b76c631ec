// The flat scan on the 16-bit matrix unit (flat_half.hip): launch interface for flat.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace qvh {

constexpr uint32_t kHalfMaxDp = 128;      // register-resident query width
constexpr uint32_t kHalfGroupRows = 16;   // rows per listed group
constexpr uint32_t kHalfTileRows = 64;
constexpr uint32_t kHalfWideTileRows = 256;    // rows wider than kHalfMaxDp: 256 rows x 256 queries
constexpr uint32_t kHalfWideQueries = 256;     // per work-group
constexpr uint32_t kHalfWideMaxDp = 4096;
constexpr uint32_t kHalfMaxLists = 512;   // lists per query the merge takes
constexpr uint32_t kHalfMaxSel = 64;      // groups the merge selects per query at most
// Batches up to which the merge takes each query with four waves (whole searches, four waves -> one:
// 600 queries, 5,000 x 768, k = 43 380 -> 545 us, 20,000 x 136, k = 11 175 -> 191 us; 1,000 queries
// over 20,000 x 136, k = 22 213 -> 192 us; 2,000 over 768 dims, k = 10, the merge alone 226 -> 194 us).
constexpr uint32_t kHalfMergeFour = 768;
// The scan's words per query in `words`: word 0 the shared bound, kHalfScaleWord the query's scale (float
// bits, written by the prep kernel). The stride keeps every query's words on lines of their own.
constexpr uint32_t kHalfWordStride = 64;
constexpr uint32_t kHalfScaleWord = 1;

/// The largest stored norm, from the store's meta words ([0] the largest squared norm, [2] the largest
/// magnitude, both float bits). Where the square is subnormal in float or has lost its bits to zero
/// (norms below 2^-50 here), the bound sqrt(dp) times the largest magnitude instead.
__device__ __forceinline__ double stored_norm(const uint32_t* meta, uint32_t dp) {
  const float n2 = __uint_as_float(meta[0]);
  return n2 < 0x1p-100f ? sqrt(static_cast<double>(dp)) * static_cast<double>(__uint_as_float(meta[2]))
                        : sqrt(static_cast<double>(n2));
}

/// 2^(11 - e) for a norm in (2^(e - 1), 2^e] (1 for zero and non-finite ones): brings the norm to
/// (2^10, 2^11]. Within 2^100 either way: smaller norms stay below it, and what they lose in 16 bits
/// is below 2^-89 times the other operand's norm, itself below 2^64.
__device__ __forceinline__ float half_scale(double norm) {
  if (!(norm > 0.0) || !(norm < __builtin_huge_val())) return 1.0f;
  int e = 0;
  const double m = frexp(norm, &e);  // m in [0.5, 1)
  if (m == 0.5) --e;
  e = 11 - e;
  return ldexpf(1.0f, e < -100 ? -100 : e > 100 ? 100 : e);
}

/// The scale of a query of norm P against a store of largest norm R. L2: the norm step's weight
/// 2^8 s_q / s_x stays within fp16 (a zero query takes its upper end: at 1 the weight would be 0 for rows
/// of norms below 2^-22, and nothing could be certified).
__device__ __forceinline__ float half_query_scale(double P, double R, bool l2) {
  const float sx = half_scale(R), sq = half_scale(P);
  return l2 && (P == 0.0 || sq > 128.0f * sx) ? 128.0f * sx : sq;
}

/// The bound on |scan's distance - reference's| for a query of norm P over rows of norms up to R, unless
/// every sum is exact: form 0 is the fp32 scans', 1 and 2 the 16-bit scans' up to kHalfMaxDp and above.
/// prep_queries_kernel derives it.
__device__ __forceinline__ double scan_bound(int form, uint32_t dp, bool l2, double P, double R) {
  const double u = 1.0 / 16777216.0;
  const double coef = (form == 2 ? 3.5 * dp + 64.0 : form == 1 ? 1.25 * dp + 64.0 : 4.0 * dp + 16.0) * u;
  return l2 ? coef * (P + R) * (P + R) + (dp + 32.0) * 0x1p-149 : coef * (1.0 + P * R);
}

struct HalfScanArgs {
  const float* X;          // [rows][dp] rows as stored (or the contiguous copy of listed rows)
  const float* xnorm;      // [rows] ||x||^2 (L2)
  uint64_t n;              // rows scanned
  uint32_t dp;             // row width: a multiple of 8 in [16, 128], for the wide form of 16 up to kHalfWideMaxDp
  const float* Q;          // [nq][dp] prepared queries
  const float* qnorm;      // [nq] ||q||^2
  uint32_t nq;
  const uint64_t* bitmap;  // admitted rows, or null
  int l2;
  uint32_t nsplit;
  uint32_t qblocks;
  uint64_t rows_per_split;  // a multiple of kHalfTileRows
  // Waves sharing each query group: 1 (every wave takes whole tiles), or 2 (the waves w and w + 4 hold
  // the same queries and take the two 32-row halves of every tile).
  uint32_t row_waves;
  float* part_d;     // [nq][lists][KL] group minima as distances, ascending
  uint32_t* part_r;  // their groups (rows 16 g .. 16 g + 15)
  uint32_t* words;   // kHalfWordStride words per query
  int share;            // 0: every list keeps its own KL best
  uint32_t share_rank;  // nonzero: the shared bound is the larger of the lane pair's entries of this rank
  const uint32_t* meta;  // the store's meta words (stored_norm)
  // The launch runs when (*gate != 0) == (gate_want != 0); null: always (the wide form takes none).
  const uint32_t* gate;
  uint32_t gate_want;
  const void* qfrag;  // wide rows: the split queries (launch_half_query_frags)
};

struct HalfMergeArgs {
  const float* X;  // the store
  uint32_t dim, dp;
  uint64_t n;  // rows scanned (positions in the list when idx is set)
  const float* Q;
  uint32_t nq, k;
  int l2;
  uint32_t nlists, sel;  // lists per query, groups selected (kl, or more for the wide merge)
  int wide;              // a list all of whose entries were taken sends the query to the exact kernel
  const float* part_d;
  const uint32_t* part_r;
  const uint32_t* idx;     // list positions -> rows, or null
  const uint64_t* bitmap;  // admitted rows, or null
  uint32_t* out_rows;
  float* out_dist;
  const float* delta;
  uint32_t* fallback;
  uint32_t* nfallback;
  const uint32_t* gate;
  uint32_t gate_want;
};

/// Queries per work-group and lists per (query, split) of a scan with lists of kl groups.
/// pair: a lane pair holds each query (two lists); otherwise one lane does.
inline uint32_t half_queries_per_block(bool pair, uint32_t row_waves) { return (pair ? 256u : 512u) / row_waves; }
inline uint32_t half_lists_per_split(bool pair) { return pair ? 2u : 1u; }

/// One scan launch. kl: 10, 16 or 32 (32 only with `pair`). products: 1 (every operand exact in
/// 16 bits) or 3.
void launch_half_scan(int kl, int products, bool pair, dim3 grid, const HalfScanArgs& a, hipStream_t s);

/// Rows wider than kHalfMaxDp (dp a multiple of 16): bytes of the split queries, the kernel that writes
/// them, and the scan (lists of 16 or 32 groups, two per query and split).
inline uint64_t half_wide_steps(uint32_t dp) { return (dp + 31) / 32 * 2; }  // 16-dim steps, whole 32-dim chunks
inline size_t half_query_frag_bytes(uint64_t nq, uint32_t dp) { return ceil_div(nq, 32) * half_wide_steps(dp) * 2048; }
void launch_half_query_frags(const float* Q, uint32_t nq, uint32_t dp, const uint32_t* words, void* out,
                             hipStream_t s);
void launch_half_wide_scan(int kl, dim3 grid, const HalfScanArgs& a, hipStream_t s);

void launch_half_merge(int kl, const HalfMergeArgs& m, hipStream_t s);

}  // namespace qvh
