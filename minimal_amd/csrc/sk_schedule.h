// sk_schedule.h -- how a stream-K launch shares S key slots out over its
// workgroups (m2l_mfma.hip).  Plain arithmetic, for the device and for host
// code: a launch and the sum over its segments must agree on it.
#pragma once
#include <cstdint>

#ifndef __HIPCC__
#define XF_HD
#else
#define XF_HD __host__ __device__
#endif

namespace xf {

// Workgroups of W that take slots: with fewer slots than workgroups some would
// have none, lie between two that do, and leave the segments unwritten that
// the sum reads from the first to the last workgroup of a tile.
XF_HD inline int sk_active(int64_t W, int64_t S) { return int(W < S ? W : S); }

// First slot of workgroup w of W active ones (W <= S: each has at least one).
XF_HD inline int64_t sk_slot(int64_t w, int64_t S, int64_t W) { return w * S / W; }

// The workgroup that takes a slot: the largest w with sk_slot(w) <= slot.
XF_HD inline int sk_owner(int64_t slot, int64_t S, int64_t W) { return int(((slot + 1) * W - 1) / S); }

}  // namespace xf
