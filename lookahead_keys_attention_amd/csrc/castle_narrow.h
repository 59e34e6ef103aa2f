// The kernels of castle_narrow.hip and the rules that choose them.
#pragma once
#include "castle_params.h"
#include <hip/hip_runtime.h>

namespace castle {

int launch_scan_narrow(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream);
int launch_attn_narrow(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream);
int launch_bwd_narrow(const BwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream);

// How many workgroups of 128 rows the wide kernels make of a shape.  The card has 256 CUs; the lines below lie where the
// two kinds crossed when both were timed at 17 shapes, 2 to 128 heads of 96 to 4096 rows (us, wide / narrow, with that
// number in front):
//   scan, bf16     96: 25 / 18    128: 43 / 29    192 (d = 128): 100 / 103    256: 28 / 29    384: 17 / 27    1024: 57 / 95
//         fp32    128: 86 / 65    192: 138 / 114  1024: 355 / 680
//   attn, d <= 64  96: 52 / 22    224: 37 / 19    256: 54 / 35   384: 28 / 25   512: 249 / 180   1024: 98 / 113
//         d = 128  16: 40 / 20    192: 200 / 135  512: 210 / 235
//   key + query    96: 115 / 90   128: 211 / 158  192 (d = 128): 536 / 445   224: 92 / 75   256: 126 / 151   1024: 354 / 635
//         fp32     16: 142 / 61   128: 1133 / 297   1024: 6488 / 3990
constexpr int kNarrowCus = 256;
inline int64_t wide_groups(const CoreShape& s) { return (int64_t)(s.Lp / 128) * s.B * s.H; }
// up to three quarters of the CUs: the wide scan's chain of blocks is halved, for twice the gates
inline bool narrow_scan(const CoreShape& s) { return wide_groups(s) <= kNarrowCus * 3 / 4; }
// up to two workgroups per CU (one at d = 128): the wide kernel has no second one to fill the waits of the first
inline bool narrow_attn(const CoreShape& s) { return wide_groups(s) <= kNarrowCus * (s.d > 64 ? 1 : 2); }
// while CUs would stay idle; fp32 at any size, as long as its score tiles are kept: the wide fp32 kernels form the scores
// once more in the query kernel, on matrix instructions an eighth as fast
inline bool narrow_bwd(const CoreShape& s, int dtype) { return dtype == 0 || wide_groups(s) < kNarrowCus; }

}  // namespace castle
