// wm_debug.h -- what the tests reach that no program needs: conditions that a
// run meets only by bad luck (a solve that cannot run side by side, a launch
// that fails) forced from the host, and counters.  Not part of the interface.
#pragma once

struct wm_ctx;

enum {
  // CUs that solves in flight hold on the device; value is added (a test that
  // plants some takes them back)
  WM_DEBUG_SOLVE_SLOTS = 1,
  // the next value on-chip solves fail to launch
  WM_DEBUG_SOLVE_FAILS = 2,
  // the next value on-chip solves wait for nothing and are taken to have given up
  WM_DEBUG_SOLVE_GIVES_UP = 3,
  // solves to come that stream; value -1 ends that
  WM_DEBUG_SOLVE_REST = 4,
  // the next on-chip solve's first tag, if value is not 0
  WM_DEBUG_SOLVE_TAG = 5,
  // slots of the largest species plane the FP64 push addresses by 32-bit byte
  // offsets, if value is not 0
  WM_DEBUG_PLANE32 = 6,
  // pinned buffers of the host arrays' copies
  WM_DEBUG_XFER_BUFFERS = 7,
};

// The quantity, after value has been put in place; -1 for an unknown key.
extern "C" long long wm_debug(wm_ctx *ctx, int key, long long value);

// wm_solve.hip's part
long long wm_debug_slots(wm_ctx *ctx, int add);
