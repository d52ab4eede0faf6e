// The LDS box of the baseline-layout degridding (bl.hip): plain C++, shared by
// the kernel and its host test.
#pragma once

constexpr int BL_BOX = 600;  // cells per wavefront: 19 KiB a workgroup

// Cells from one box row to the next: odd, so that rows start on different banks.
constexpr int bl_box_pitch(int bw) { return bw | 1; }

// Whether windows spanning bw x bh cells fit the box.  Each extent can be the
// whole grid's (65536), whose product no int holds: rows past the box's cells
// count as one more than these.
constexpr bool bl_box_fits(int bw, int bh) {
  return (bh < BL_BOX + 1 ? bh : BL_BOX + 1) * bl_box_pitch(bw) <= BL_BOX;
}
