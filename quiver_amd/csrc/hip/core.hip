// Process-wide state of the qvh library: error reporting, device selection, the allocation
// fault hook, and row normalization.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <string>

#include "common.hpp"
#include "exact.hpp"

namespace qvh {
namespace {

thread_local std::string t_last_error;

std::mutex g_device_mu;
int g_device = -1;     // device chosen by qvh_init (or 0 on first use)
bool g_checked = false;

std::atomic<long> g_alloc_count{0};
long fault_alloc_at() {
  static const long at = [] {
    const char* s = std::getenv("QVH_FAULT_ALLOC");
    return s && *s ? std::atol(s) : 0L;
  }();
  return at;
}

void check_device(int dev) {
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
    throw Failure(QVH_EDEVICE, "no HIP device is available (the qvh kernels need a gfx950 GPU)");
  }
  if (dev < 0 || dev >= count) {
    throw Failure(QVH_EINVAL, "device " + std::to_string(dev) + " does not exist (" +
                                  std::to_string(count) + " HIP devices)");
  }
  hipDeviceProp_t prop;
  QVH_HIP(hipGetDeviceProperties(&prop, dev));
  if (std::string(prop.gcnArchName).rfind("gfx950", 0) != 0) {
    throw Failure(QVH_EDEVICE, std::string("device is ") + prop.gcnArchName +
                                   "; the qvh kernels are built for gfx950 only");
  }
}

// simd::normalize (src/simd/dispatch.cc:119-135) of every row in place, eight lanes per row: the
// group computes the row's dot product in the reference's order (exact_group8, bit for bit as
// exact_dot), every lane then scales its share of the row by the same 1/sqrt(norm^2). A non-finite
// sum takes the double-precision redo in the group's first lane, as exact_normalize does.
__global__ void normalize_rows_kernel(float* __restrict__ rows, uint64_t n, uint32_t dim) {
  const uint64_t t = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t r = t >> 3;
  const uint32_t l = static_cast<uint32_t>(t & 7u);
  const bool valid = r < n;
  float* v = rows + (valid ? r : 0) * dim;
  const float lead = exact_group8<false>(v, v, dim, valid);  // every lane of the wave takes part
  const float norm_sq = __shfl(lead, 0, 8);
  if (!valid) return;
  if (!isfinite(norm_sq)) {
    if (l == 0) exact_normalize(v, dim);
    return;
  }
  if (norm_sq <= 0.0f) return;
  const float inv = 1.0f / sqrtf(norm_sq);
  for (uint32_t i = l; i < dim; i += 8) v[i] = v[i] * inv;
}

/// Raises *flag (host memory the device can write) when some value is not finite.
__global__ void __launch_bounds__(256) finite_kernel(const float* __restrict__ x, uint64_t n, uint32_t* flag) {
  bool ok = true;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * 256) {
    ok = ok && isfinite(x[i]);
  }
  if (__builtin_amdgcn_ballot_w64(!ok) != 0 && (threadIdx.x & 63) == 0) {
    __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__global__ void __launch_bounds__(256) map_rows_kernel(const uint32_t* __restrict__ rows, uint64_t count,
                                                       const uint64_t* __restrict__ table, uint64_t n,
                                                       int64_t* __restrict__ out) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= count) return;
  const uint32_t r = rows[i];
  out[i] = r < n ? static_cast<int64_t>(table[r]) : -1;
}

__global__ void __launch_bounds__(256) map_refs_kernel(const uint64_t* __restrict__ refs, uint64_t count,
                                                       const uint64_t* __restrict__ offsets, uint64_t nlist,
                                                       const uint64_t* __restrict__ table, uint64_t n,
                                                       int64_t* __restrict__ out) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= count) return;
  const uint64_t ref = refs[i], list = ref >> 32;
  const uint64_t pos = list < nlist ? offsets[list] + (ref & 0xFFFFFFFFull) : n;
  out[i] = ref != QVH_EMPTY_REF && pos < n ? static_cast<int64_t>(table[pos]) : -1;
}

/// One word of pinned host memory per thread that checks device inputs, released when it ends.
struct PinnedWord {
  uint32_t* ptr = nullptr;
  PinnedWord() = default;
  PinnedWord(const PinnedWord&) = delete;
  PinnedWord& operator=(const PinnedWord&) = delete;
  ~PinnedWord() {
    if (ptr) (void)hipHostFree(ptr);
  }
  uint32_t* get() {
    if (!ptr) {
      void* p = nullptr;
      QVH_HIP(hipHostMalloc(&p, sizeof(uint32_t), hipHostMallocPortable));
      ptr = static_cast<uint32_t*>(p);
    }
    return ptr;
  }
};
thread_local PinnedWord t_finite;

}  // namespace

void set_last_error(const std::string& msg) { t_last_error = msg; }

int current_device() {
  std::lock_guard<std::mutex> lock(g_device_mu);
  if (g_device < 0) g_device = 0;
  if (!g_checked) {
    check_device(g_device);
    g_checked = true;
  }
  QVH_HIP(hipSetDevice(g_device));
  return g_device;
}

void* device_alloc(size_t bytes) {
  const long n = ++g_alloc_count;
  if (fault_alloc_at() > 0 && n == fault_alloc_at()) {
    throw Failure(QVH_ENOMEM, "injected allocation failure (QVH_FAULT_ALLOC=" +
                                  std::to_string(n) + ")");
  }
  void* p = nullptr;
  QVH_HIP(hipMalloc(&p, bytes == 0 ? 1 : bytes));
  return p;
}

void device_free(void* p) noexcept {
  // Asynchronous work of any stream may still read a buffer that is regrown or released: the
  // device finishes it first.
  if (p) {
    (void)hipDeviceSynchronize();
    (void)hipFree(p);
  }
}

void launch_normalize_rows(float* d_rows, uint64_t n, uint32_t dim, hipStream_t stream) {
  if (n == 0) return;
  const unsigned block = 256;  // 32 rows
  hipLaunchKernelGGL(normalize_rows_kernel, dim3(static_cast<unsigned>(ceil_div(n * 8, block))),
                     dim3(block), 0, stream, d_rows, n, dim);
  QVH_HIP(hipGetLastError());
}

}  // namespace qvh

extern "C" {

const char* qvh_last_error(void) { return qvh::t_last_error.c_str(); }

qvh_status qvh_device_allocations(uint64_t* count) {
  if (count == nullptr) {
    qvh::set_last_error("qvh_device_allocations: null output");
    return QVH_EINVAL;
  }
  *count = static_cast<uint64_t>(qvh::g_alloc_count.load());
  return QVH_OK;
}

qvh_status qvh_init(int device) {
  return qvh::guarded([&] {
    std::lock_guard<std::mutex> lock(qvh::g_device_mu);
    qvh::check_device(device);
    qvh::g_device = device;
    qvh::g_checked = true;
    QVH_HIP(hipSetDevice(device));
  });
}

qvh_status qvh_get_device(int* device) {
  return qvh::guarded([&] {
    QVH_REQUIRE(device != nullptr, "qvh_get_device: null argument");
    *device = qvh::current_device();
  });
}

qvh_status qvh_device_info(char* name, size_t name_len, char* arch, size_t arch_len,
                           int* compute_units) {
  return qvh::guarded([&] {
    const int dev = qvh::current_device();
    hipDeviceProp_t prop;
    QVH_HIP(hipGetDeviceProperties(&prop, dev));
    if (name && name_len) {
      std::strncpy(name, prop.name, name_len - 1);
      name[name_len - 1] = '\0';
    }
    if (arch && arch_len) {
      std::strncpy(arch, prop.gcnArchName, arch_len - 1);
      arch[arch_len - 1] = '\0';
    }
    if (compute_units) *compute_units = prop.multiProcessorCount;
  });
}

qvh_status qvh_device_finite(const float* d_x, uint64_t count, void* stream, int* finite) {
  return qvh::guarded([&] {
    QVH_REQUIRE(finite != nullptr, "qvh_device_finite: null output");
    *finite = 1;
    if (count == 0) return;
    QVH_REQUIRE(d_x != nullptr, "qvh_device_finite: null buffer");
    qvh::current_device();
    uint32_t* flag = qvh::t_finite.get();
    __atomic_store_n(flag, 0u, __ATOMIC_RELEASE);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const uint64_t blocks = std::min<uint64_t>(qvh::ceil_div(count, 1024), 1024);
    hipLaunchKernelGGL(qvh::finite_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, d_x, count, flag);
    QVH_HIP(hipGetLastError());
    QVH_HIP(hipStreamSynchronize(s));
    *finite = __atomic_load_n(flag, __ATOMIC_ACQUIRE) == 0u ? 1 : 0;
  });
}

qvh_status qvh_upload(void* d_dst, const void* src, uint64_t bytes, void* stream) {
  return qvh::guarded([&] {
    if (bytes == 0) return;
    QVH_REQUIRE(d_dst && src, "qvh_upload: null buffer");
    qvh::current_device();
    const hipStream_t s = static_cast<hipStream_t>(stream);
    QVH_HIP(hipMemcpyAsync(d_dst, src, bytes, hipMemcpyHostToDevice, s));
    QVH_HIP(hipStreamSynchronize(s));
  });
}

qvh_status qvh_map_rows_device(const uint32_t* d_rows, uint64_t count, const uint64_t* d_table, uint64_t n,
                               int64_t* d_labels, void* stream) {
  return qvh::guarded([&] {
    if (count == 0) return;
    QVH_REQUIRE(d_rows && d_table && d_labels && stream, "qvh_map_rows_device: null argument");
    qvh::current_device();
    hipLaunchKernelGGL(qvh::map_rows_kernel, dim3(static_cast<unsigned>(qvh::ceil_div(count, 256))), dim3(256), 0,
                       static_cast<hipStream_t>(stream), d_rows, count, d_table, n, d_labels);
    QVH_HIP(hipGetLastError());
  });
}

qvh_status qvh_map_refs_device(const uint64_t* d_refs, uint64_t count, const uint64_t* d_offsets, uint64_t nlist,
                               const uint64_t* d_table, uint64_t n, int64_t* d_labels, void* stream) {
  return qvh::guarded([&] {
    if (count == 0) return;
    QVH_REQUIRE(d_refs && d_offsets && d_table && d_labels && stream, "qvh_map_refs_device: null argument");
    qvh::current_device();
    hipLaunchKernelGGL(qvh::map_refs_kernel, dim3(static_cast<unsigned>(qvh::ceil_div(count, 256))), dim3(256), 0,
                       static_cast<hipStream_t>(stream), d_refs, count, d_offsets, nlist, d_table, n, d_labels);
    QVH_HIP(hipGetLastError());
  });
}

qvh_status qvh_normalize(float* rows, uint64_t n, uint32_t dim) {
  return qvh::guarded([&] {
    QVH_REQUIRE(rows != nullptr || n == 0, "qvh_normalize: null rows");
    QVH_REQUIRE(dim >= 1, "qvh_normalize: dim must be positive");
    if (n == 0) return;
    qvh::current_device();
    qvh::DeviceBuffer buf;
    const size_t bytes = static_cast<size_t>(n) * dim * sizeof(float);
    float* d = static_cast<float*>(buf.reserve(bytes));
    QVH_HIP(hipMemcpy(d, rows, bytes, hipMemcpyHostToDevice));
    qvh::launch_normalize_rows(d, n, dim, nullptr);
    QVH_HIP(hipMemcpy(rows, d, bytes, hipMemcpyDeviceToHost));
  });
}

}  // extern "C"
