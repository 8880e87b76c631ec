// What the flat scan's bound rests on, for tests/test_flat_half_bound_gpu.py: single matrix steps, and the
// group minima that the 16-bit scans list, with the bound the search uses for them. Calls the scans of
// libqvh.so through their launch interface.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "flat_half.hpp"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

/// One wave per tile: d = a b + c with a [32][16], b [32][16] (a column of the product per row), c, d [32][32].
__global__ void __launch_bounds__(64) matrix_step_kernel(const _Float16* a, const _Float16* b, const float* c, float* d) {
  const int j = threadIdx.x & 31, h = threadIdx.x >> 5;
  const size_t t = blockIdx.x;
  const f16x8 x = *reinterpret_cast<const f16x8*>(a + t * 512 + j * 16 + 8 * h);
  const f16x8 y = *reinterpret_cast<const f16x8*>(b + t * 512 + j * 16 + 8 * h);
  f32x16 acc;
  for (int r = 0; r < 16; ++r) acc[r] = c[t * 1024 + (8 * (r / 4) + 4 * h + r % 4) * 32 + j];
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, y, acc, 0, 0, 0);
  for (int r = 0; r < 16; ++r) d[t * 1024 + (8 * (r / 4) + 4 * h + r % 4) * 32 + j] = acc[r];
}

/// The queries' scales, bounds and shared words, as the search's own preparation of them.
__global__ void prepare_kernel(const double* norms, uint32_t nq, uint32_t dp, int l2, int form, const uint32_t* meta,
                               uint32_t* words, double* bound) {
  const uint32_t q = blockIdx.x * 64 + threadIdx.x;
  if (q >= nq) return;
  const double R = qvh::stored_norm(meta, dp);
  for (uint32_t i = 0; i < qvh::kHalfWordStride; ++i) words[q * qvh::kHalfWordStride + i] = 0xFF800000u;
  words[q * qvh::kHalfWordStride + qvh::kHalfScaleWord] = __float_as_uint(qvh::half_query_scale(norms[q], R, l2 != 0));
  bound[q] = qvh::scan_bound(form, dp, l2 != 0, norms[q], R);
}

struct Buffers {
  std::vector<void*> held;
  bool ok = true;
  template <class T>
  T* get(size_t count, const T* from = nullptr) {
    void* p = nullptr;
    ok = ok && hipMalloc(&p, count * sizeof(T)) == hipSuccess;
    if (ok) held.push_back(p);
    if (ok && from) ok = hipMemcpy(p, from, count * sizeof(T), hipMemcpyHostToDevice) == hipSuccess;
    return static_cast<T*>(p);
  }
  template <class T>
  void put(T* to, const T* from, size_t count) {
    ok = ok && hipMemcpy(to, from, count * sizeof(T), hipMemcpyDeviceToHost) == hipSuccess;
  }
  ~Buffers() {
    for (void* p : held) (void)hipFree(p);
  }
};

}  // namespace

extern "C" int probe_matrix_steps(const uint16_t* a, const uint16_t* b, const float* c, float* d, uint32_t tiles) {
  Buffers m;
  const uint16_t *da = m.get(size_t{tiles} * 512, a), *db = m.get(size_t{tiles} * 512, b);
  const float* dc = m.get(size_t{tiles} * 1024, c);
  float* dd = m.get<float>(size_t{tiles} * 1024);
  if (!m.ok || tiles == 0) return 1;
  hipLaunchKernelGGL(matrix_step_kernel, dim3(tiles), dim3(64), 0, nullptr, reinterpret_cast<const _Float16*>(da),
                     reinterpret_cast<const _Float16*>(db), dc, dd);
  m.ok = hipGetLastError() == hipSuccess;
  m.put(d, dd, size_t{tiles} * 1024);
  return m.ok ? 0 : 1;
}

/// Group minima of x [n][dp] (n a multiple of rows_per_split, every split's groups fitting its lists) for q
/// [nq][dp]: minima and groups [nq][lists][kl], lists by split, and the bounds [nq]. xnorm and qnorm are
/// the squared norms as floats, qlen the queries' norms, meta the store's words.
extern "C" int probe_half_minima(const float* x, const float* xnorm, uint64_t n, uint32_t dp, const float* q,
                                 const float* qnorm, const double* qlen, uint32_t nq, int l2, const uint32_t* meta, int kl,
                                 int products, int pair, uint64_t rows_per_split, float* minima, uint32_t* groups,
                                 double* bound) {
  const bool wide = dp > qvh::kHalfMaxDp;
  const uint32_t per_split = wide ? 2 : qvh::half_lists_per_split(pair != 0);
  const uint64_t tile = wide ? qvh::kHalfWideTileRows : qvh::kHalfTileRows;
  if (n == 0 || nq == 0 || n % rows_per_split || rows_per_split % tile || dp % (wide ? 16 : 8) || dp < 16 ||
      dp > qvh::kHalfWideMaxDp) {
    return 2;
  }
  const uint32_t nsplit = static_cast<uint32_t>(n / rows_per_split);
  const size_t entries = size_t{nq} * nsplit * per_split * kl;
  Buffers m;
  qvh::HalfScanArgs a{};
  a.X = m.get(n * dp, x);
  a.xnorm = m.get(n, xnorm);
  a.n = n;
  a.dp = dp;
  a.Q = m.get(size_t{nq} * dp, q);
  a.qnorm = m.get(nq, qnorm);
  a.nq = nq;
  a.l2 = l2;
  a.nsplit = nsplit;
  a.rows_per_split = rows_per_split;
  a.row_waves = 1;
  a.part_d = m.get<float>(entries);
  a.part_r = m.get<uint32_t>(entries);
  a.words = m.get<uint32_t>(size_t{nq} * qvh::kHalfWordStride);
  a.meta = m.get(4, meta);
  const double* dlen = m.get(nq, qlen);
  double* db = m.get<double>(nq);
  void* frags = wide ? m.get<unsigned char>(qvh::half_query_frag_bytes(nq, dp)) : nullptr;
  if (!m.ok) return 1;
  hipLaunchKernelGGL(prepare_kernel, dim3((nq + 63) / 64), dim3(64), 0, nullptr, dlen, nq, dp, l2, wide ? 2 : 1, a.meta,
                     a.words, db);
  const uint32_t per_block = wide ? qvh::kHalfWideQueries : qvh::half_queries_per_block(pair != 0, 1);
  a.qblocks = (nq + per_block - 1) / per_block;
  const dim3 grid(a.qblocks * nsplit);
  if (wide) {
    qvh::launch_half_query_frags(a.Q, nq, dp, a.words, frags, nullptr);
    a.qfrag = frags;
    qvh::launch_half_wide_scan(kl, grid, a, nullptr);
  } else {
    qvh::launch_half_scan(kl, products, pair != 0, grid, a, nullptr);
  }
  m.ok = hipGetLastError() == hipSuccess;
  m.put(minima, a.part_d, entries);
  m.put(groups, a.part_r, entries);
  m.put(bound, db, nq);
  return m.ok ? 0 : 1;
}
