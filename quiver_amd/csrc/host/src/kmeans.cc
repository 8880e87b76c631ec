#include <algorithm>
#include <cstring>
#include <memory>
#include <numeric>
#include <random>
#include <type_traits>

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

/// Points in one cluster up to which an iteration takes its means on the device. There one wave adds a
/// cluster's points one after another, 45 ns a point (78 past 64 dims), so the largest cluster decides;
/// the host adds every point once, one thread per 8 dims and sub-space. The bits are the same.
/// Nanoseconds a point and iteration, assignment included (four iterations of random points, host and
/// device at k = 4, 16, 64, 256):
///   65,536 points     4 dims  3.2, 12.7   2.9, 6.0   2.8, 3.4   3.2, 2.9
///                    16 dims  5.4, 18.2   4.9, 7.6   5.0, 4.5   6.6, 4.1
///                    64 dims  8.6, 22.0   7.9, 9.4    10, 6.5   8.9, 5.6
///                   128 dims   19, 32      19, 16     20, 12     20, 9.3
///   500,000          16 dims  4.2, 15     3.9, 7.0   4.0, 3.9   5.1, 2.8
///                    64 dims   26, 19      23, 8.8    22, 5.8    22, 5.4
/// (At these sizes 1 dim is the host's at every k up to 256, 2 dims up to 512; with points past the
/// host's caches its sums wait for memory.) Past 256 centroids a dimension the device's reads of every assignment
/// per centroid are left to the host's sums too.
std::size_t device_means_limit(std::size_t n, std::size_t nsub, std::size_t dsub, std::size_t k) {
  if (k > 256 * dsub || n >= 0xFFFFFFFFull) return 0;
  const double points = static_cast<double>(n), dims = static_cast<double>(dsub);
  const bool cached = points * dims * static_cast<double>(nsub) * sizeof(float) <= 48e6;
  // 40 us an iteration for the copy down and the threads' start (2,000 x 16, k = 8, 20 iterations: 1.0 ms on
  // the device, 1.9 on the host).
  const double each = dsub <= 8 ? 1.2 + 0.35 * dims : cached ? 3.5 + 0.12 * dims : 18.0 + 0.08 * dims;
  const double host_ns = static_cast<double>(nsub) * each + 40e3 / points;
  const double device_ns = 1.7 + (dsub <= 8 ? 0.0 : 0.06 * dims);
  const double even = (host_ns - device_ns) / (dsub <= 64 ? 45.0 : 78.0);
  // Past 8 dims more than the break-even: a first iteration's clusters are the least even ones, and the
  // host loses the more the fewer its threads.
  const double lenient = dsub <= 8 ? 1.0 : !cached ? 1.5 : dsub <= 16 || dsub > 64 ? 2.0 : 3.0;
  const auto limit = static_cast<std::size_t>(std::clamp(lenient * even, 0.0, 1.0) * points);
  // Some cluster holds at least n / k points, and of many the largest about three times that.
  return points * (dsub <= 8 ? 3.0 : 1.0) > static_cast<double>(limit) * static_cast<double>(k) ? 0 : limit;
}

/// The means of the clusters with points of every sub-space into cent, counts[nsub][k] the points: each
/// (cluster, dimension) adds its points in index order, in double. `sums` is scratch.
void host_means(const float* x, std::size_t n, std::size_t dim, std::size_t nsub, std::size_t k,
                const std::uint32_t* assign, std::vector<std::size_t>& counts, std::vector<double>& sums,
                std::vector<float>& cent, ThreadPool& tp) {
  const std::size_t dsub = dim / nsub, chunks = (dsub + 7) / 8;
  std::fill(counts.begin(), counts.end(), std::size_t{0});
  for (std::size_t s = 0; s < nsub; ++s) {
    for (std::size_t i = 0; i < n; ++i) ++counts[s * k + assign[s * n + i]];
  }
  const std::size_t stride = k * 8 + 8;  // by chunk and a line apart: no thread writes to another's cache lines
  sums.resize(nsub * chunks * stride);
  tp.parallel_for(nsub * chunks, 1, [&](std::size_t begin, std::size_t end) {
    for (std::size_t chunk = begin; chunk < end; ++chunk) {
      const std::size_t s = chunk / chunks, jb = chunk % chunks * 8, je = std::min(dsub, jb + 8);
      double* const sum = sums.data() + chunk * stride;
      std::fill(sum, sum + k * 8, 0.0);
      for (std::size_t i = 0; i < n; ++i) {
        const float* const v = x + i * dim + s * dsub;
        double* const to = sum + static_cast<std::size_t>(assign[s * n + i]) * 8;
        for (std::size_t j = jb; j < je; ++j) to[j - jb] += static_cast<double>(v[j]);
      }
      for (std::size_t c = 0; c < k; ++c) {
        const std::size_t count = counts[s * k + c];
        if (count == 0) continue;
        float* const mean = cent.data() + (s * k + c) * dsub;
        for (std::size_t j = jb; j < je; ++j) mean[j] = static_cast<float>(sum[c * 8 + j - jb] / static_cast<double>(count));
      }
    }
  });
}

/// Lloyd iterations for nsub sub-spaces at once, each with its own centroids in cent
/// [nsub][k][dim / nsub] and its own draws: assignment on the device, means there or on the host
/// (device_means_limit; an iteration that meets a larger cluster ends on the host, and so do the next
/// ones while it stays so).
void lloyd(const float* x, std::size_t n, std::size_t dim, std::size_t nsub, std::size_t k, std::size_t iterations,
           std::vector<std::mt19937_64>& rng, std::vector<float>& cent, ThreadPool& tp) {
  if (iterations == 0) return;
  qvh_points* raw = nullptr;
  internal::qvh_check(qvh_points_create(x, n, static_cast<std::uint32_t>(dim), &raw), "kmeans");
  std::unique_ptr<qvh_points, PointsDeleter> points(raw);
  const std::size_t dsub = dim / nsub;
  const std::size_t most = device_means_limit(n, nsub, dsub, k);
  std::size_t limit = most;
  const auto install = [&] {
    internal::qvh_check(qvh_points_set_centroids(points.get(), cent.data(), static_cast<std::uint32_t>(k),
                                                 static_cast<std::uint32_t>(nsub)),
                        "kmeans centroids");
  };
  const auto fetch = [&] { internal::qvh_check(qvh_points_get_centroids(points.get(), cent.data()), "kmeans centroids"); };
  install();
  bool fetched = true;  // cent holds the installed centroids
  std::vector<std::uint32_t> device_counts(nsub * k), assign;
  std::vector<std::size_t> host_counts;
  std::vector<double> sums;
  for (std::size_t iter = 0; iter < iterations; ++iter) {
    const bool last = iter + 1 == iterations;
    int stepped = 0;
    internal::qvh_check(qvh_points_step_within(points.get(), static_cast<std::uint32_t>(limit), device_counts.data(),
                                               &stepped),
                        "kmeans step");
    // Splits the empty clusters of an iteration and installs what the host has changed.
    const auto finish = [&](auto& counts, bool changed) {
      using Count = typename std::decay_t<decltype(counts)>::value_type;
      const bool empty = std::find(counts.begin(), counts.end(), Count{0}) != counts.end();
      if (!fetched && (last || empty)) {
        fetch();
        fetched = true;
      }
      if (empty) {
        for (std::size_t s = 0; s < nsub; ++s) {
          split_empty_clusters(cent.data() + s * k * dsub, counts.data() + s * k, k, dsub, n, rng[s]);
        }
      }
      if (!last && (changed || empty)) install();
    };
    if (stepped != 0) {
      fetched = false;
      finish(device_counts, false);
    } else {
      if (!fetched) fetch();
      fetched = true;
      assign.resize(nsub * n);
      host_counts.resize(nsub * k);
      internal::qvh_check(qvh_points_assigned(points.get(), assign.data()), "kmeans assignment");
      host_means(x, n, dim, nsub, k, assign.data(), host_counts, sums, cent, tp);
      limit = *std::max_element(host_counts.begin(), host_counts.end()) > most ? 0 : most;
      finish(host_counts, true);
    }
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

}  // namespace

namespace internal {

std::vector<float> kmeans_subspaces(const float* vectors, std::size_t n, std::size_t dim, std::size_t nsub,
                                    const KMeansParams& params, ThreadPool* pool) {
  const std::size_t k = params.k, dsub = dim / nsub;
  std::vector<float> cent(nsub * k * dsub);
  std::vector<std::mt19937_64> rng;
  std::vector<std::size_t> order(n);
  std::iota(order.begin(), order.end(), std::size_t{0});
  for (std::size_t s = 0; s < nsub; ++s) {
    rng.emplace_back(params.seed + s);
    draw_initial(vectors, dim, s * dsub, dsub, k, order, rng.back(), cent.data() + s * k * dsub);
  }
  lloyd(vectors, n, dim, nsub, k, params.iterations, rng, cent, pool ? *pool : ThreadPool::global());
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
  std::vector<std::mt19937_64> one{rng};
  lloyd(x, n, dim, 1, k, params.iterations, one, cent, pool ? *pool : ThreadPool::global());
  return cent;
}

}  // namespace quiver
