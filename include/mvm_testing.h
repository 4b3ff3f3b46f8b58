/*
 * mvm_testing.h -- test hooks of libmvm_scan.so.  Not part of the drop-in
 * boundary and with no counterpart in the reference; the test suite uses them
 * to check the lane layout of the cross-lane reductions on the device, and on
 * the host which columns a kernel reads.
 */
#ifndef MVM_TESTING_H
#define MVM_TESTING_H

#ifdef __cplusplus
extern "C" {
#endif

/* One wave: lane l holds x_j = 1000*j + l (j = 0..3).  Writes 128 floats to
 * device memory `out`: [0,64) the 4-lane state-group sum of x_0 per lane,
 * [64,128) the 16-channel reduction of (x_0..x_3) per lane. */
int mvm_selftest_lanes(float* out, void* stream);

/* Host only: the columns of a dt row that mvm_scan_fused_dt_fwd reads for a
 * dt rank, 16 per staging group, as the kernel forms them; at most 48 are
 * written to `cols`.  Returns their number, or < 0 for a bad rank. */
int mvm_selftest_dt_columns(int dt_rank, int* cols);

#ifdef __cplusplus
}
#endif

#endif /* MVM_TESTING_H */
