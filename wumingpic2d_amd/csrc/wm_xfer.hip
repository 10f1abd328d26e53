// wm_xfer.hip -- host arrays to and from the device.
//
// A copy between the device and memory that the runtime has not pinned goes
// through its own staging buffer on one thread, and a destination whose pages
// have not been touched yet is faulted in page by page on the way: 30 MB take
// 1.8 ms (2.9 into fresh pages), of which the link needs 0.56.  Here up to
// eight threads each own a pinned buffer and take pieces of the array in turn:
// while one waits for its piece the others copy theirs, and a destination's
// pages are touched while its piece is on the way.  202 MB of fields in pieces of
// 4 MB: 11.7 -> 4.7 ms.  Arrays below 64 MB go up in pieces of 2 MB (58 MB 1.9 ms,
// by the runtime 14.7) and down in pieces of 1 MB, as fast as 2 MB and the buffers
// made sooner: 30 MB of moments on 512 x 512 with 64 per cell and species, a
// context's first call 2.7 ms, later ones 1.9; by the runtime 3.1 and 2.95, with
// eight buffers of 2 MB and the runtime's copies 3.4 and, by turns, 2.0 and 3.6.
// Arrays below 8 MB go by one thread with two buffers of 1 MB.
//
// Rows of particles are gathered from and scattered to the caller's arrays in
// the same pass; they used to go through a vector of the whole state, zeroed,
// filled and copied on one thread (35 MB of rows in an array of 176: 9.7 -> 1.1
// ms).
//
// The threads live as long as the call; the pinned buffers (1 to 4 MB each,
// made when first needed) as long as the context.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <numeric>
#include <system_error>
#include <thread>

#include "wm_internal.h"
#include "wm_xfer.h"

namespace {
// The largest piece of a copy, and the size of the buffers it needs.
size_t slot_for(size_t bytes, bool up) {
  constexpr size_t MB = (size_t)1 << 20;
  return bytes < 8 * MB ? MB : bytes < 64 * MB ? (up ? 2 * MB : MB) : 4 * MB;
}
constexpr int WORKERS = 8;
// Threads for a copy: one up to 8 MB, then one per MB.  Starting one costs
// about 20 us, and now and then milliseconds where the process has used up its
// share of the processors (its other threads may be waiting actively); 5 MB by
// one thread take 0.30 ms, as by four.
int threads_for(size_t bytes) {
  constexpr size_t ALONE = (size_t)8 << 20, SHARE = (size_t)1 << 20;
  return bytes < ALONE ? 1 : (int)std::min<size_t>(WORKERS, bytes / SHARE);
}

// The buffers a copy may make anew, beyond `few`.  One of 1 MB takes 0.05 to 0.15
// ms, and the process makes one at a time, so that eight cost a context's first
// copies of a few MB more than eight threads save: a state of 9 MB goes up in
// 1.4 ms by the runtime's staging, 1.8 with eight new buffers, 1.1 with two.  Two
// serve it as well as eight, later too.
int new_buffers(size_t bytes) {
  constexpr size_t MB = (size_t)1 << 20;
  return bytes < 16 * MB ? 0 : (int)((bytes - 8 * MB) >> 22);
}

// Threads with a buffer each that a copy has at once.  Down four: the caller's
// pages, often fresh ones, are touched and filled on the way.  A moments call whose
// result is 15.5 MB takes 1.05 ms by four, 1.18 by two and 1.15 by eight and the
// runtime's copies; two steps and 12.6 MB of particles to the host 0.72, 0.87 and
// 0.90.  Eight would give 0.02 more, for four calls of 0.3 more to make their
// buffers.
int few(bool up) { return up ? 2 : 4; }

// f(worker) on `n` threads, the caller's as worker 0; fewer if the system
// gives no more.
template <class F>
void on_threads(int n, F f) {
  std::vector<std::thread> t;
  t.reserve(n);
  try {
    for (int k = 1; k < n; ++k) t.emplace_back([&f, k] { f(k); });
  } catch (const std::system_error &) {
  }
  f(0);
  for (std::thread &x : t) x.join();
}
}  // namespace

struct wm_xfer {
  void *pin[WORKERS] = {};
  size_t size[WORKERS] = {};
  hipEvent_t ev[WORKERS] = {};
  bool busy[WORKERS] = {};                     // the device may still read it
};

void wm_xfer_free(wm_ctx *ctx) {
  if (!ctx->xfer) return;
  for (int k = 0; k < WORKERS; ++k) {
    if (ctx->xfer->pin[k]) (void)hipHostFree(ctx->xfer->pin[k]);
    if (ctx->xfer->ev[k]) (void)hipEventDestroy(ctx->xfer->ev[k]);
  }
  delete ctx->xfer;
  ctx->xfer = nullptr;
}

int wm_xfer_buffers(const wm_ctx *ctx) {
  int n = 0;
  if (ctx->xfer)
    for (size_t s : ctx->xfer->size) n += s > 0;
  return n;
}

namespace {
// Buffer k, of `size` bytes at least and not in use.
hipError_t slot_of(wm_xfer &x, int k, size_t size) {
  hipError_t e = hipSuccess;
  if (!x.ev[k]) e = hipEventCreateWithFlags(&x.ev[k], hipEventDisableTiming);
  if (e == hipSuccess && x.busy[k]) {
    e = hipEventSynchronize(x.ev[k]);
    x.busy[k] = e != hipSuccess;
  }
  if (e != hipSuccess || x.size[k] >= size) return e;
  if (x.pin[k]) e = hipHostFree(x.pin[k]);
  x.pin[k] = nullptr;
  x.size[k] = 0;
  if (e == hipSuccess) e = hipHostMalloc(&x.pin[k], size, hipHostMallocCoherent);
  if (e == hipSuccess) x.size[k] = size;
  return e;
}

struct Chunk {
  size_t s0, s1;                            // pieces
};

// n bytes (both ends on 8-byte boundaries) to a pinned buffer.  Copies that the
// runtime is asked for while others are on their way go to several DMA engines:
// making one's queue takes a millisecond of a context's first call, and some
// move 12 GB/s where others move 41, so that 30 MB took 1.5 ms in two calls of
// three and 3.1 in the third.  By this kernel 1.4 to 1.6 ms.  (Uploads have shown
// neither, and from new buffers a kernel reads more slowly than they.)
// One array of more than a piece by one thread (`plain`) stays with the runtime,
// whose copies then follow one another: a moments call of 5.5 MB 0.48 to 0.50 ms,
// by the kernel 0.50 to 0.53.  Arrays of several parts and single pieces are faster
// by the kernel: two steps and 6.3 MB of particles to the host 0.52 ms, by the
// runtime 0.57.
__global__ __launch_bounds__(256) void k_to_pinned(const char *src, char *dst, size_t n) {
  const double *s = (const double *)src;
  double *d = (double *)dst;
  const size_t n8 = n / 8, st = (size_t)gridDim.x * 256;
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * st < n8; i += 4 * st) {
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = s[i + k * st];
#pragma unroll
    for (int k = 0; k < 4; ++k) d[i + k * st] = v[k];
  }
  for (; i < n8; i += st) d[i] = s[i];
  if (blockIdx.x == 0 && threadIdx.x < n % 8) dst[8 * n8 + threadIdx.x] = src[8 * n8 + threadIdx.x];
}
hipError_t to_pinned(char *pin, const char *dev, size_t n, hipStream_t st, bool plain) {
  if (plain || (size_t)dev % 8 != 0) return hipMemcpyAsync(pin, dev, n, hipMemcpyDeviceToHost, st);
  const size_t blocks = std::max<size_t>(1, std::min<size_t>(64, n / 2048));
  hipLaunchKernelGGL(k_to_pinned, dim3((unsigned)blocks), dim3(256), 0, st, dev, pin, n);
  return hipGetLastError();
}

// Has the pages of memory that is about to be written faulted in (their
// contents stay).
void touch(const char *p, size_t n) {
  constexpr size_t PAGE = 4096;
  if (n == 0) return;
  for (size_t o = 0; o < n; o += PAGE) {
    volatile char *q = const_cast<char *>(p) + o;
    *q = *q;
  }
  volatile char *q = const_cast<char *>(p) + n - 1;
  *q = *q;
}

int move(wm_ctx *ctx, char *dev, const std::vector<WmSpan> &spans, bool up, size_t rec, size_t keep) {
  size_t total = 0;
  for (const WmSpan &s : spans) total += s.bytes;
  if (total == 0) return WM_OK;
  if (!ctx->xfer) ctx->xfer = new wm_xfer;
  wm_xfer &x = *ctx->xfer;
  const size_t slot = slot_for(total, up);
  int have = 0;
  for (size_t s : x.size) have += s >= slot;
  const int want = std::min(threads_for(total), std::max(few(up), have + new_buffers(total)));
  // (one thread alone has two buffers, and copies a chunk while the next is on
  // its way)
  const bool plain = want == 1 && spans.size() == 1 && total > slot;
  const size_t unit = std::lcm(rec, (size_t)16);
  const size_t most = std::min(slot, std::max<size_t>(total / want + rec, (size_t)1 << 20)) / unit * unit;
  std::vector<WmSpan> piece;
  std::vector<Chunk> chunk;
  for (const WmSpan &s : spans)
    for (size_t o = 0; o < s.bytes; o += most)
      piece.push_back({s.host + o, s.at + o, std::min(most, s.bytes - o)});
  for (size_t k = 0; k < piece.size();) {
    size_t e = k + 1;
    while (e < piece.size() && piece[e].at + piece[e].bytes - piece[k].at <= most) ++e;
    chunk.push_back({k, e});
    k = e;
  }
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  hipStream_t st = ctx->stream;
  const int device = ctx->device;
  on_threads((int)std::min<size_t>(want, chunk.size()), [&](int w) {
    hipError_t e = w > 0 ? hipSetDevice(device) : hipSuccess;   // (a thread's own)
    size_t last = chunk.size();               // down: the chunk on its way
    const int other = want > 1 ? 0 : 1;
    int buf = w;
    auto land = [&](size_t c, int b) {        // chunk c, in buffer b, to its place
      const Chunk &h = chunk[c];
      for (size_t k = h.s0; k < h.s1; ++k) touch(piece[k].host, piece[k].bytes);
      const hipError_t r = hipEventSynchronize(x.ev[b]);
      if (r != hipSuccess) return r;
      x.busy[b] = false;
      for (size_t k = h.s0; k < h.s1; ++k) {
        char *d = const_cast<char *>(piece[k].host);
        const char *s = (const char *)x.pin[b] + (piece[k].at - piece[h.s0].at);
        if (keep == rec) {
          memcpy(d, s, piece[k].bytes);
        } else {
          for (size_t o = 0; o < piece[k].bytes; o += rec) memcpy(d + o, s + o, keep);
        }
      }
      return r;
    };
    for (size_t c; e == hipSuccess && err.load() == (int)hipSuccess && (c = next++) < chunk.size();) {
      const Chunk &h = chunk[c];
      const size_t at = piece[h.s0].at, len = piece[h.s1 - 1].at + piece[h.s1 - 1].bytes - at;
      e = slot_of(x, buf, slot);
      if (e != hipSuccess) break;
      x.busy[buf] = true;
      char *pin = (char *)x.pin[buf];
      if (up) {
        for (size_t k = h.s0; k < h.s1; ++k) memcpy(pin + (piece[k].at - at), piece[k].host, piece[k].bytes);
        e = hipMemcpyAsync(dev + at, pin, len, hipMemcpyHostToDevice, st);
      } else {
        e = to_pinned(pin, dev + at, len, st, plain);
      }
      if (e == hipSuccess) e = hipEventRecord(x.ev[buf], st);
      if (e == hipSuccess && !up) {
        if (other == 0) e = land(c, buf);
        else if (last < chunk.size()) e = land(last, buf ^ 1);
        last = c;
      }
      buf ^= other;
    }
    if (!up && other && e == hipSuccess && last < chunk.size()) e = land(last, buf ^ 1);
    int ok = (int)hipSuccess;
    if (e != hipSuccess) err.compare_exchange_strong(ok, (int)e);
  });
  WM_HIP((hipError_t)err.load());
  return WM_OK;
}
}  // namespace

int wm_to_device(wm_ctx *ctx, void *dev, const std::vector<WmSpan> &spans) {
  return move(ctx, (char *)dev, spans, true, 1, 1);
}
int wm_to_host(wm_ctx *ctx, const void *dev, const std::vector<WmSpan> &spans, size_t rec,
               size_t keep) {
  return move(ctx, (char *)const_cast<void *>(dev), spans, false, rec, keep);
}
int wm_to_device(wm_ctx *ctx, void *dev, const void *host, size_t bytes) {
  return wm_to_device(ctx, dev, {{(const char *)host, 0, bytes}});
}
int wm_to_host(wm_ctx *ctx, const void *dev, void *host, size_t bytes) {
  return wm_to_host(ctx, dev, {{(const char *)host, 0, bytes}}, 1, 1);
}

void wm_touch(void *host, size_t bytes) {
  const int n = threads_for(bytes);
  on_threads(n, [&](int k) {
    const size_t a = bytes * k / n, b = bytes * (k + 1) / n;
    touch((const char *)host + a, b - a);
  });
}

void wm_copy_field6(double *dst, const double *src, const int *from, size_t np, int nrow) {
  const size_t bytes = (size_t)nrow * np * 96;
  const int want = threads_for(bytes / 2);
  std::atomic<int> next{0};
  on_threads(std::min(want, nrow), [&](int) {
    for (int s; (s = next++) < nrow;)
      for (size_t k = (size_t)s * np + from[s]; k < (size_t)(s + 1) * np; ++k) dst[6 * k + 5] = src[6 * k + 5];
  });
}
