"""The test suite's way to what no program needs (csrc/wm_debug.h)."""
import ctypes

SOLVE_SLOTS = 1      # CUs held by solves in flight on the device; value is added
SOLVE_FAILS = 2      # on-chip solves that fail to launch
SOLVE_GIVES_UP = 3   # on-chip solves that wait for nothing and give up
SOLVE_REST = 4       # solves to come that stream (-1 ends that)
SOLVE_TAG = 5        # the next on-chip solve's first tag (if not 0)
PLANE32 = 6          # largest plane the FP64 push addresses in 32 bits (if not 0)
XFER_BUFFERS = 7     # pinned buffers of the host arrays' copies


def debug(ctx, key, value=0):
    f = ctx._lib.wm_debug
    f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_int, ctypes.c_longlong], ctypes.c_longlong
    return f(ctx._h, key, value)
