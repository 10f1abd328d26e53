// wm_order.h -- the code the FP64 push leaves per particle for the row order
// (wm_order.hip): bits 2..15 the new cell (0-based column, below 2^14), bits
// 0..1 what becomes of it.
#pragma once

enum : unsigned {
  WM_CODE_STAY = 0,    // stays in its row, at most one cell away
  WM_CODE_UP = 1,      // to the row above
  WM_CODE_DOWN = 2,    // to the row below
  WM_CODE_FAR = 3      // stays in its row, more than one cell away
};
