#include <algorithm>
#include <cstring>
#include <memory>
#include <numeric>
#include <random>

#include "device_util.h"
#include "quiver/quantizer.h"

namespace quiver {

namespace {
struct PointsDeleter {
  void operator()(qvh_points* p) const noexcept { qvh_points_destroy(p); }
};

/// Splits every empty cluster of k x dim centroids off a donor drawn with probability proportional
/// to its size (src/product_quantizer.cc:101-117).
template <class Count>
void split_empty_clusters(float* cent, Count* counts, std::size_t k, std::size_t dim, std::size_t n,
                          std::mt19937_64& rng) {
  for (std::size_t c = 0; c < k; ++c) {
    if (counts[c] != 0) continue;
    std::size_t donor = 0;
    for (;;) {
      donor = rng() % k;
      const double share = static_cast<double>(counts[donor]) / static_cast<double>(n) * static_cast<double>(k);
      if (share > std::uniform_real_distribution<double>(0.0, 1.0)(rng)) break;
    }
    constexpr float kEps = 1.0f / 1024.0f;
    for (std::size_t j = 0; j < dim; ++j) {
      const float v = cent[donor * dim + j];
      const float sign = (j % 2 == 0) ? 1.0f : -1.0f;
      cent[c * dim + j] = v * (1.0f + sign * kEps);
      cent[donor * dim + j] = v * (1.0f - sign * kEps);
    }
    counts[c] = counts[donor] / 2;
    counts[donor] -= counts[c];
  }
}

/// Lloyd iterations with the assignment and the means on the device, for nsub sub-spaces at once
/// (each with its own centroids in cent [nsub][k][dim / nsub] and its own draws). The host sees the
/// counts of each iteration, and the centroids when some cluster is empty.
void lloyd_on_device(const float* x, std::size_t n, std::size_t dim, std::size_t nsub, std::size_t k,
                     std::size_t iterations, std::vector<std::mt19937_64>& rng, std::vector<float>& cent) {
  if (iterations == 0) return;
  qvh_points* raw = nullptr;
  internal::qvh_check(qvh_points_create(x, n, static_cast<std::uint32_t>(dim), &raw), "kmeans");
  std::unique_ptr<qvh_points, PointsDeleter> points(raw);
  const std::size_t dsub = dim / nsub;
  const auto install = [&] {
    internal::qvh_check(qvh_points_set_centroids(points.get(), cent.data(), static_cast<std::uint32_t>(k),
                                                 static_cast<std::uint32_t>(nsub)),
                        "kmeans centroids");
  };
  install();
  std::vector<std::uint32_t> counts(nsub * k);
  for (std::size_t iter = 0; iter < iterations; ++iter) {
    internal::qvh_check(qvh_points_step(points.get(), counts.data()), "kmeans step");
    const bool last = iter + 1 == iterations;
    const bool empty = std::find(counts.begin(), counts.end(), 0u) != counts.end();
    if (!last && !empty) continue;
    internal::qvh_check(qvh_points_get_centroids(points.get(), cent.data()), "kmeans centroids");
    if (!empty) continue;
    for (std::size_t s = 0; s < nsub; ++s) {
      split_empty_clusters(cent.data() + s * k * dsub, counts.data() + s * k, k, dsub, n, rng[s]);
    }
    if (!last) install();
  }
}

/// k distinct points drawn by a partial Fisher-Yates over [0, n) (src/product_quantizer.cc:53-62):
/// columns [off, off + dsub) of each into cent. `order` is [0, n) in order, and is left so.
void draw_initial(const float* x, std::size_t dim, std::size_t off, std::size_t dsub, std::size_t k,
                  std::vector<std::size_t>& order, std::mt19937_64& rng, float* cent) {
  const std::size_t n = order.size();
  std::vector<std::size_t> touched(k);
  for (std::size_t i = 0; i < k; ++i) {
    touched[i] = i + rng() % (n - i);
    std::swap(order[i], order[touched[i]]);
    std::memcpy(cent + i * dsub, x + order[i] * dim + off, dsub * sizeof(float));
  }
  for (std::size_t i = k; i-- > 0;) std::swap(order[i], order[touched[i]]);
}

/// The device reads every assignment once per centroid, the host adds dim values per point: past 256
/// centroids a dimension the host's sums are the cheaper ones (by the memory rates of both sides;
/// every product-quantizer sub-space, with 256 centroids, is on the device's side).
bool means_on_device(std::size_t k, std::size_t dim) { return k <= 256 * dim; }
}  // namespace

namespace internal {

std::vector<float> kmeans_subspaces(const float* vectors, std::size_t n, std::size_t dim, std::size_t nsub,
                                    const KMeansParams& params) {
  const std::size_t k = params.k, dsub = dim / nsub;
  std::vector<float> cent(nsub * k * dsub);
  std::vector<std::mt19937_64> rng;
  std::vector<std::size_t> order(n);
  std::iota(order.begin(), order.end(), std::size_t{0});
  for (std::size_t s = 0; s < nsub; ++s) {
    rng.emplace_back(params.seed + s);
    draw_initial(vectors, dim, s * dsub, dsub, k, order, rng.back(), cent.data() + s * k * dsub);
  }
  lloyd_on_device(vectors, n, dim, nsub, k, params.iterations, rng, cent);
  return cent;
}

}  // namespace internal

// Steps and random draws as in the reference's kmeans (src/product_quantizer.cc:29-117), which
// the bit-identical result requires: subsample by a partial Fisher-Yates over rng() % (n - i),
// initialize from k distinct points the same way, then per iteration assign (on the device),
// average in double, and split each empty cluster off a donor drawn with probability
// proportional to its size.
std::vector<float> kmeans(const float* vectors, std::size_t n, std::size_t dim,
                          const KMeansParams& params, ThreadPool* pool) {
  const std::size_t k = params.k;
  QUIVER_CHECK(k > 0 && dim > 0, "kmeans: k and dim must be positive");
  QUIVER_CHECK(n >= k, "kmeans: need at least k=" + std::to_string(k) + " training points, got " +
                           std::to_string(n));
  QUIVER_CHECK(k <= 0xFFFFFFFFull && dim <= 0xFFFFFFFFull, "kmeans: k or dim too large");
  ThreadPool& tp = pool ? *pool : ThreadPool::global();
  std::mt19937_64 rng(params.seed);

  const float* x = vectors;
  std::vector<float> sample;
  const std::size_t cap = k * std::max<std::size_t>(1, params.max_points_per_centroid);
  if (n > cap) {
    std::vector<std::size_t> order(n);
    std::iota(order.begin(), order.end(), std::size_t{0});
    for (std::size_t i = 0; i < cap; ++i) std::swap(order[i], order[i + rng() % (n - i)]);
    sample.resize(cap * dim);
    for (std::size_t i = 0; i < cap; ++i) {
      std::memcpy(sample.data() + i * dim, vectors + order[i] * dim, dim * sizeof(float));
    }
    x = sample.data();
    n = cap;
  }

  std::vector<float> cent(k * dim);
  {
    std::vector<std::size_t> order(n);
    std::iota(order.begin(), order.end(), std::size_t{0});
    draw_initial(x, dim, 0, dim, k, order, rng, cent.data());
  }
  if (means_on_device(k, dim) && n < 0xFFFFFFFFull) {
    std::vector<std::mt19937_64> one{rng};
    lloyd_on_device(x, n, dim, 1, k, params.iterations, one, cent);
    return cent;
  }

  qvh_points* raw = nullptr;
  internal::qvh_check(qvh_points_create(x, n, static_cast<std::uint32_t>(dim), &raw), "kmeans");
  std::unique_ptr<qvh_points, PointsDeleter> points(raw);

  std::vector<std::uint32_t> assign(n);
  std::vector<double> sums(k * dim);
  std::vector<std::size_t> counts(k);
  for (std::size_t iter = 0; iter < params.iterations; ++iter) {
    internal::qvh_check(qvh_points_nearest(points.get(), cent.data(), static_cast<std::uint32_t>(k), 0,
                                           assign.data()),
                        "kmeans assignment");
    std::fill(counts.begin(), counts.end(), std::size_t{0});
    for (std::size_t i = 0; i < n; ++i) ++counts[assign[i]];
    // Per (cluster, dimension) the points are added in index order; chunks split dimensions.
    tp.parallel_for(dim, 8, [&](std::size_t jb, std::size_t je) {
      for (std::size_t c = 0; c < k; ++c)
        for (std::size_t j = jb; j < je; ++j) sums[c * dim + j] = 0.0;
      for (std::size_t i = 0; i < n; ++i) {
        const std::size_t c = assign[i];
        for (std::size_t j = jb; j < je; ++j) sums[c * dim + j] += static_cast<double>(x[i * dim + j]);
      }
    });
    for (std::size_t c = 0; c < k; ++c) {
      if (counts[c] == 0) continue;
      for (std::size_t j = 0; j < dim; ++j) {
        cent[c * dim + j] = static_cast<float>(sums[c * dim + j] / static_cast<double>(counts[c]));
      }
    }
    split_empty_clusters(cent.data(), counts.data(), k, dim, n, rng);
  }
  return cent;
}

}  // namespace quiver
