// vx_stage.h -- a call's host operands and results cross the bus through
// pinned memory that a small kernel on the engine's stream reads or writes.
// hipMemcpyAsync on the caller's pageable memory costs the host 10-20 us a copy
// (its own staging, and a wait for each copy back), which a small call pays two
// to five times: a two-layer step at 3900 positions took 144 us for 110 us of
// kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

namespace vx {

constexpr size_t STAGE_BYTES = (size_t)1 << 20;  // each way; larger operands are copied by hipMemcpyAsync
typedef uint32_t st_u32x4 __attribute__((ext_vector_type(4)));

// bytes: a multiple of 4; both addresses are 16-byte aligned
__global__ __launch_bounds__(256) void stage_copy_kernel(const uint32_t *src, uint32_t *dst, int bytes) {
  const int i = 4 * (blockIdx.x * 256 + threadIdx.x), left = bytes / 4 - i;
  if (left >= 4) *(st_u32x4 *)(dst + i) = *(const st_u32x4 *)(src + i);
  else
    for (int q = 0; q < left; q++) dst[i + q] = src[i + q];
}

// One call's operands and results in the engine's staging memory (host address
// h, device address d: [0, STAGE_BYTES) in, then as much out), which the next
// call reuses.  finish() waits for the stream and hands the results over; a
// call that returns before it, on an error, waits in the destructor, so that
// nothing queued still reads or writes the memory, or a caller's buffer, when
// the next call fills it.
class Stage {
 public:
  Stage(hipStream_t st, unsigned char *h, unsigned char *d) : st_(st), h_(h), d_(d) {}
  Stage(const Stage &) = delete;
  Stage &operator=(const Stage &) = delete;
  ~Stage() {
    if (pending_) (void)hipStreamSynchronize(st_);
  }
  // for a kernel that uses the staging memory itself: called before its launch
  void hold() { pending_ = true; }

  hipError_t in(void *dev, const void *src, size_t bytes) {
    if (bytes == 0) return hipSuccess;
    pending_ = true;
    if (bytes % 4 || in_at_ + bytes > STAGE_BYTES) return hipMemcpyAsync(dev, src, bytes, hipMemcpyHostToDevice, st_);
    memcpy(h_ + in_at_, src, bytes);
    copy(dev, d_ + in_at_, bytes);
    in_at_ += (bytes + 255) & ~(size_t)255;
    return hipSuccess;
  }
  hipError_t out(void *dst, const void *dev, size_t bytes) {
    if (bytes == 0) return hipSuccess;
    pending_ = true;
    if (n_ == 4 || bytes % 4 || ((uintptr_t)dev & 15) || out_at_ + bytes > STAGE_BYTES)
      return hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, st_);
    const size_t at = STAGE_BYTES + out_at_;
    copy(d_ + at, dev, bytes);
    outs_[n_++] = {dst, at, bytes};
    out_at_ += (bytes + 255) & ~(size_t)255;
    return hipSuccess;
  }
  hipError_t finish() {
    hipError_t s = hipGetLastError();
    if (s == hipSuccess) s = hipStreamSynchronize(st_);
    if (s != hipSuccess) return s;
    pending_ = false;
    for (int i = 0; i < n_; i++) memcpy(outs_[i].dst, h_ + outs_[i].at, outs_[i].bytes);
    return hipSuccess;
  }

 private:
  void copy(void *dst, const void *src, size_t bytes) {
    hipLaunchKernelGGL(stage_copy_kernel, dim3((bytes + 4095) / 4096), dim3(256), 0, st_, (const uint32_t *)src,
                       (uint32_t *)dst, (int)bytes);
  }
  struct Out {
    void *dst;
    size_t at, bytes;
  };
  hipStream_t st_;
  unsigned char *h_, *d_;
  bool pending_ = false;  // the stream may hold work on the staging memory
  size_t in_at_ = 0, out_at_ = 0;
  int n_ = 0;
  Out outs_[4] = {};
};

}  // namespace vx
