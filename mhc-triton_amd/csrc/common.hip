// Host-side plumbing shared by every entry point: error reporting and device
// queries.
#include <stdarg.h>
#include <stdio.h>

#include "common.hpp"

namespace mhc {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int hip_status(hipError_t e, const char* where) {
  if (e == hipSuccess) return MHC_OK;
  set_error("%s: %s", where, hipGetErrorString(e));
  return MHC_ERR_HIP;
}

int num_cus() {
  static thread_local int dev_cached = -1;
  static thread_local int cus = 256;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return cus;
  if (dev != dev_cached) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) cus = v;
    dev_cached = dev;
  }
  return cus;
}

}  // namespace mhc

namespace mhc {

// mhc_convert: a thread per element over the concatenated segments (end[i]: where segment i ends).
// Bound by its launch: the largest segment, phi, is 1.5 MB at dim 4096.  One launch for a module's
// parameters in place of a conversion kernel each: 3 + 6 of the static layer's training step and
// 7 + 14 of the dynamic layer's, about 4 us of GPU time and 4 us of host time apiece.
struct ConvertArgs {
  const void* src[MHC_CONVERT_MAX];
  void* dst[MHC_CONVERT_MAX];
  int64_t end[MHC_CONVERT_MAX];
  int sd[MHC_CONVERT_MAX], dd[MHC_CONVERT_MAX];
  int n;
};

__global__ __launch_bounds__(kThreads) void convert_kernel(ConvertArgs a) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  int64_t beg = 0;
#pragma unroll
  for (int k = 0; k < MHC_CONVERT_MAX; ++k) {
    if (k >= a.n) return;
    if (i < a.end[k]) {
      const int64_t e = i - beg;
      const float v = a.sd[k] == MHC_DTYPE_F32    ? static_cast<const float*>(a.src[k])[e]
                      : a.sd[k] == MHC_DTYPE_BF16 ? to_f32(static_cast<const __bf16*>(a.src[k])[e])
                                                  : to_f32(static_cast<const _Float16*>(a.src[k])[e]);
      if (a.dd[k] == MHC_DTYPE_F32) static_cast<float*>(a.dst[k])[e] = v;
      else if (a.dd[k] == MHC_DTYPE_BF16) static_cast<__bf16*>(a.dst[k])[e] = from_f32<__bf16>(v);
      else static_cast<_Float16*>(a.dst[k])[e] = from_f32<_Float16>(v);
      return;
    }
    beg = a.end[k];
  }
}

}  // namespace mhc

extern "C" int mhc_convert(int n, const void* const* src, const int* src_dtype, void* const* dst, const int* dst_dtype,
                           const int64_t* count, mhc_stream_t stream) {
  using namespace mhc;
  if (n < 0 || n > MHC_CONVERT_MAX || (n && (!src || !src_dtype || !dst || !dst_dtype || !count))) {
    set_error("convert: %d tensors (at most %d) or a null array", n, MHC_CONVERT_MAX);
    return MHC_ERR_ARG;
  }
  ConvertArgs a{};
  int64_t total = 0;
  for (int i = 0; i < n; ++i) {
    if (count[i] < 0 || (count[i] && (!src[i] || !dst[i]))) {
      set_error("convert: bad count or null pointer (tensor %d)", i);
      return MHC_ERR_ARG;
    }
    for (int dt : {src_dtype[i], dst_dtype[i]})
      if (dt != MHC_DTYPE_F32 && dt != MHC_DTYPE_BF16 && dt != MHC_DTYPE_F16) {
        set_error("unsupported dtype code %d", dt);
        return MHC_ERR_DTYPE;
      }
    total += count[i];
    a.src[i] = src[i];
    a.dst[i] = dst[i];
    a.sd[i] = src_dtype[i];
    a.dd[i] = dst_dtype[i];
    a.end[i] = total;
  }
  a.n = n;
  if (total == 0) return MHC_OK;
  if (total > ((int64_t)1 << 31) * kThreads - kThreads) {
    set_error("convert: %lld elements", (long long)total);
    return MHC_ERR_ARG;
  }
  convert_kernel<<<dim3((unsigned)((total + kThreads - 1) / kThreads)), kThreads, 0, (hipStream_t)stream>>>(a);
  return hip_status(hipGetLastError(), "convert launch");
}

extern "C" int mhc_abi_version(void) { return 3; }

extern "C" const char* mhc_last_error(void) { return mhc::g_err; }
