// Vertex arrays between host (interleaved x y [z] per vertex, float or
// double) and device (one array per component, the handle's real type).
//
// The bound is the host's own copy (about 10 GB/s a core; the link takes
// 50), so the host touches every byte once: it copies the caller's array
// into pinned slots in slices (checking it for non-finite values on the
// way), and one kernel per slice reads the pinned slot over the link,
// converts and splits the components through LDS, in 16-byte words on the
// link side and whole lines on the device side.  Downloads run the same way
// back.  Two slots alternate, so host copy and link overlap; arrays of 8 MB
// and more are copied by four threads (each with two slots), below that a
// thread's start costs more than it saves.  2.65 M float vertices (32 MB): up
// 10.1 -> 3.4 ms, back 10.3 -> 3.5 ms with the first touch of a fresh result
// array; 9 x 162 vertices: a call of upload, one step and three reads
// 196 -> 120 us.
#pragma once

#include <thread>

constexpr int kXferVerts = 1024;              // vertices per workgroup
constexpr size_t kXferSlot = 512u << 10;      // bytes of a pinned slot
constexpr size_t kXferThreaded = 8u << 20;    // bytes from which four threads copy
constexpr int kXferThreads = 4;

struct XferSlots {
  unsigned char* host = nullptr;
  size_t slot = 0;
  int n = 0;
  hipEvent_t ev[2 * kXferThreads] = {};
  bool pending[2 * kXferThreads] = {};
  void release() {
    for (int i = 0; i < n; i++)
      if (pending[i]) (void)hipEventSynchronize(ev[i]);
    for (hipEvent_t& e : ev) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (host) (void)hipHostFree(host);
    host = nullptr;
    n = 0;
    slot = 0;
    for (bool& p : pending) p = false;
  }
};

// One slice of vertices, at most a slot: grid of kXferVerts per workgroup.
// lo (may be null): the float residuals of the positions, component stride
// lo_stride.  The last 16-byte word may reach past the slice, not past the
// slot (its size is a multiple of 16).
template <typename H, typename R, int NC>
__global__ void __launch_bounds__(256) k_split(const H* src, R* c0, R* c1, R* c2, float* lo, size_t lo_stride, int n) {
  __shared__ uint4 buf[kXferVerts * NC * sizeof(H) / 16];
  const int i0 = blockIdx.x * kXferVerts, cnt = min(kXferVerts, n - i0);
  const uint4* in = reinterpret_cast<const uint4*>(src + (size_t)i0 * NC);
  const int words = (cnt * NC * (int)sizeof(H) + 15) / 16;
  for (int w = threadIdx.x; w < words; w += 256) buf[w] = in[w];
  __syncthreads();
  const H* v = reinterpret_cast<const H*>(buf);
  for (int i = threadIdx.x; i < cnt; i += 256) {
    c0[i0 + i] = (R)v[NC * i];
    c1[i0 + i] = (R)v[NC * i + 1];
    if (NC == 3) c2[i0 + i] = (R)v[NC * i + 2];
    if (lo)  // what the float positions did not keep
      for (int k = 0; k < NC; k++)
        lo[k * lo_stride + i0 + i] = (float)((double)v[NC * i + k] - (double)(float)v[NC * i + k]);
  }
}

template <typename H, typename R, int NC>
__global__ void __launch_bounds__(256) k_merge(H* dst, const R* c0, const R* c1, const R* c2, const float* lo,
                                               size_t lo_stride, int n) {
  __shared__ uint4 buf[kXferVerts * NC * sizeof(H) / 16];
  const int i0 = blockIdx.x * kXferVerts, cnt = min(kXferVerts, n - i0);
  H* v = reinterpret_cast<H*>(buf);
  for (int i = threadIdx.x; i < cnt; i += 256) {
    const R p[3] = {c0[i0 + i], c1[i0 + i], NC == 3 ? c2[i0 + i] : R(0)};
    for (int k = 0; k < NC; k++) {
      H q = (H)p[k];
      if (lo) q += (H)lo[k * lo_stride + i0 + i];
      v[NC * i + k] = q;
    }
  }
  __syncthreads();
  uint4* out = reinterpret_cast<uint4*>(dst + (size_t)i0 * NC);
  const int words = (cnt * NC * (int)sizeof(H) + 15) / 16;
  for (int w = threadIdx.x; w < words; w += 256) out[w] = buf[w];
}

// Copies n values and tells whether all of them are finite (the exponent
// bits; a plain loop the compiler can vectorise).
template <typename T>
static bool copy_finite(T* dst, const T* src, size_t n) {
  using U = std::conditional_t<sizeof(T) == 8, unsigned long long, unsigned>;
  const U inf = sizeof(T) == 8 ? (U)0x7ff0000000000000ull : (U)0x7f800000u;
  U bad = 0;
  constexpr size_t kRun = 4096;  // checked while it is in the cache
  for (size_t a = 0; a < n; a += kRun) {
    const size_t m = std::min(kRun, n - a);
    std::memcpy(dst + a, src + a, m * sizeof(T));
    for (size_t i = 0; i < m; i++) {
      U b;
      std::memcpy(&b, src + a + i, sizeof(T));
      bad |= (U)((b & inf) == inf);
    }
  }
  return bad == 0;
}
