// lh_xfer.hpp -- fields between the device layout [plane][column] and the host's f(j, column).
//
// The layouts are transposes of each other.  The device transposes into (or out of) a staging
// area in its own memory, and the staged bytes cross PCIe through pinned buffers: worker threads
// take 2 MB chunks in turn, each with a buffer of its own, so that one thread's copy between its
// buffer and the caller's pageable memory overlaps the others' transfers.  A 384x289x384 state
// (1.37 GB): download 480 -> 45 ms, upload 640 -> 35 ms; the former host loops read one element
// per 1.2 MB stride, and a copy to fresh pageable memory alone runs at 10 GB/s (pinned: 57).
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace lh {

// one field: nj device planes; host rows 0 .. n - 1 are the planes j0 .. j0 + n - 1
struct XferField {
  void* dev;
  void* host;       // caller's array, null: skip
  size_t stage;     // byte offset in the staging area
  int nj, j0, n;
};
struct XferFields {
  XferField f[5];
};

constexpr int kXT = 32;
// staging [column][n] <- planes (UP false), planes <- staging (UP true; planes outside the host
// rows are cleared): 32 x 32 tiles through LDS, field blockIdx.z
template <typename T, bool UP>
__global__ void __launch_bounds__(kXT * 8) k_xfer(XferFields fs, char* stage, int ncol) {
  const XferField f = fs.f[blockIdx.z];
  __shared__ T tile[kXT][kXT + 1];
  T* const dev = reinterpret_cast<T*>(f.dev);
  T* const st = reinterpret_cast<T*>(stage + f.stage);
  const int c0 = blockIdx.x * kXT, s0 = blockIdx.y * kXT;       // columns, planes (UP) or host rows
  const int tx = threadIdx.x % kXT, ty = threadIdx.x / kXT;
  if (s0 >= (UP ? f.nj : f.n)) return;                            // uniform over the block
  if (UP) {
    for (int k = ty; k < kXT; k += 8) {
      const int r = s0 + tx - f.j0;
      T v{};
      if (c0 + k < ncol && r >= 0 && r < f.n) v = st[(size_t)(c0 + k) * f.n + r];
      tile[k][tx] = v;
    }
    __syncthreads();
    for (int k = ty; k < kXT; k += 8)
      if (s0 + k < f.nj && c0 + tx < ncol) dev[(size_t)(s0 + k) * ncol + c0 + tx] = tile[tx][k];
  } else {
    for (int k = ty; k < kXT; k += 8)
      if (s0 + k < f.n && c0 + tx < ncol) tile[k][tx] = dev[(size_t)(f.j0 + s0 + k) * ncol + c0 + tx];
    __syncthreads();
    for (int k = ty; k < kXT; k += 8)
      if (c0 + k < ncol && s0 + tx < f.n) st[(size_t)(c0 + k) * f.n + s0 + tx] = tile[tx][k];
  }
}

// The pinned memory, shared by every handle of the process and freed with the last one: per device
// the transfer buffers, allocated with its first transfer and used by one transfer at a time (its link
// to the host is the limit of concurrent ones too), and 128-byte slots, one per handle, cut from 32 KB
// slabs (an allocation per handle costs 0.3 ms).  A transfer holds its device's lock alone: handles come
// and go, and other devices transfer, while it waits.
struct HostStage {
  static constexpr size_t kChunk = 2u << 20;
  static constexpr int kThreads = 4, kSlot = 16, kSlab = 256;    // doubles per slot, slots per slab
  struct Link {
    std::mutex mu;
    char* buf = nullptr;
  };
  std::mutex mu;                          // of the members below
  int users = 0;
  std::map<int, Link> links;              // by device (an entry stays where it is)
  std::vector<double*> slabs, free_slots;
  Link& link(int dev) {
    std::lock_guard<std::mutex> g(mu);
    return links[dev];
  }
  // a slot for a new handle (null: no pinned memory)
  double* retain() {
    std::lock_guard<std::mutex> g(mu);
    if (free_slots.empty()) {
      double* s = nullptr;
      if (hipHostMalloc((void**)&s, sizeof(double) * kSlot * kSlab, hipHostMallocPortable | hipHostMallocMapped) !=
          hipSuccess)
        return nullptr;
      slabs.push_back(s);
      for (int i = kSlab - 1; i >= 0; --i) free_slots.push_back(s + (size_t)i * kSlot);
    }
    double* const r = free_slots.back();
    free_slots.pop_back();
    memset(r, 0, sizeof(double) * kSlot);
    ++users;
    return r;
  }
  void release(double* slot) {
    std::lock_guard<std::mutex> g(mu);
    free_slots.push_back(slot);
    if (--users > 0) return;
    for (double* s : slabs) (void)hipHostFree(s);
    slabs.clear();
    free_slots.clear();
    for (auto& l : links) {               // (no handle is left, so no transfer)
      if (l.second.buf) (void)hipHostFree(l.second.buf);
      l.second.buf = nullptr;
    }
  }
};
// (never destroyed: a host's own global may give its handle back after the statics made later are gone)
inline HostStage& host_stage() {
  static HostStage* const s = new HostStage;
  return *s;
}

// the staged bytes of nf fields (element size el, ncol columns) to or from the callers' arrays,
// in order on stream st of device dev; complete at return
inline hipError_t xfer_bytes(bool up, int dev, hipStream_t st, char* stage, const XferFields& fs, int nf, int ncol,
                             size_t el) {
  HostStage::Link& hs = host_stage().link(dev);
  std::lock_guard<std::mutex> g(hs.mu);
  if (!hs.buf) {
    const hipError_t e = hipHostMalloc((void**)&hs.buf, HostStage::kChunk * HostStage::kThreads, hipHostMallocPortable);
    if (e != hipSuccess) {
      hs.buf = nullptr;
      return e;
    }
  }
  // chunk k of the job: up to kChunk bytes of one field
  size_t first[6] = {0}, total = 0;
  for (int i = 0; i < nf; ++i) {
    const size_t bytes = fs.f[i].host ? (size_t)fs.f[i].n * ncol * el : 0;
    total += bytes;
    first[i + 1] = first[i] + (bytes + HostStage::kChunk - 1) / HostStage::kChunk;
  }
  const size_t nchunk = first[nf];
  // (a thread per chunk's worth of bytes: below that its start costs more than the copy it takes over)
  const int nt = (int)std::min<size_t>(HostStage::kThreads, 1 + total / HostStage::kChunk);
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  auto work = [&](int t) {
    char* const b = hs.buf + (size_t)t * HostStage::kChunk;
    hipEvent_t ev = nullptr;
    hipError_t e = hipSetDevice(dev);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    while (e == hipSuccess && err.load() == (int)hipSuccess) {
      const size_t k = next.fetch_add(1);
      if (k >= nchunk) break;
      int i = 0;
      while (k >= first[i + 1]) ++i;
      const size_t bytes = (size_t)fs.f[i].n * ncol * el, o = (k - first[i]) * HostStage::kChunk;
      const size_t len = std::min(HostStage::kChunk, bytes - o);
      char* const host = static_cast<char*>(fs.f[i].host) + o;
      char* const d = stage + fs.f[i].stage + o;
      if (up) memcpy(b, host, len);
      e = hipMemcpyAsync(up ? d : b, up ? b : d, len, up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipEventRecord(ev, st);
      if (e == hipSuccess) e = hipEventSynchronize(ev);
      if (e == hipSuccess && !up) memcpy(host, b, len);
    }
    if (ev) (void)hipEventDestroy(ev);
    if (e != hipSuccess) err.store((int)e);
  };
  std::thread pool[HostStage::kThreads];
  int started = 0;
  try {
    for (int t = 1; t < nt; ++t) {
      pool[t] = std::thread(work, t);
      started = t;
    }
  } catch (const std::system_error&) {
    // fewer threads than asked for: those that run take every chunk
  }
  int cur = dev;
  (void)hipGetDevice(&cur);
  work(0);
  for (int t = 1; t <= started; ++t) pool[t].join();
  if (cur != dev) (void)hipSetDevice(cur);             // the caller's device stays current
  return (hipError_t)err.load();
}

}  // namespace lh
