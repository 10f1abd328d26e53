// wm_xfer.h -- host arrays to and from the device (wm_xfer.hip).
#pragma once
#include <cstddef>
#include <vector>

struct wm_ctx;

// A piece of a host array and its place in a device buffer.
struct WmSpan {
  const char *host;
  size_t at, bytes;
};

// The spans (ascending places, none overlapping) to the device, on the
// context's stream; the host memory has been read when this returns.  The
// device bytes between two spans may be written too.
int wm_to_device(wm_ctx *ctx, void *dev, const std::vector<WmSpan> &spans);
// From the device, once the stream's earlier work is done; the host memory
// holds it when this returns, and nothing outside the spans is written.  With
// rec: records of rec bytes, of which the first keep are written.
int wm_to_host(wm_ctx *ctx, const void *dev, const std::vector<WmSpan> &spans, size_t rec = 1,
               size_t keep = 1);
// The same for one array.
int wm_to_device(wm_ctx *ctx, void *dev, const void *host, size_t bytes);
int wm_to_host(wm_ctx *ctx, const void *dev, void *host, size_t bytes);
// Has the pages of an array that a later wm_to_host fills faulted in, while the
// device works.
void wm_touch(void *host, size_t bytes);
void wm_xfer_free(wm_ctx *ctx);
int wm_xfer_buffers(const wm_ctx *ctx);   // pinned buffers it has

// Component 6 of the records from[s] .. np - 1 of every row s (np records).
void wm_copy_field6(double *dst, const double *src, const int *from, size_t np, int nrow);
