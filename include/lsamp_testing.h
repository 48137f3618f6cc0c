/*
 * lsamp_testing.h — test hooks of liblsamp.so.  Not part of the production
 * ABI: no reference counterpart, and a production caller must never call
 * anything declared here (the Swift module map does not export this header).
 */
#ifndef LSAMP_TESTING_H
#define LSAMP_TESTING_H

#include "lsamp.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The bounded waits (the fused arrangement's and the top-k kernel's
 * finalizer), process-wide on `device`: polls > 0 makes every wait's target
 * unreachable and gives it up after `polls` polls, so the fail-closed path
 * (LSAMP_ROW_TIMEOUT, token -1) runs while every kernel exits normally;
 * 0 restores normal waits.  While it is set, every fused or top-k row on the
 * device fails closed.  Synchronous; not for use while other calls are in
 * flight. */
lsamp_status lsamp_test_set_spin_limit(int32_t device, int32_t polls);

/* The launch plan of lsamp_top2 (`lse` 0) / lsamp_logprobs (1) for `rows` rows of
 * `vocab` logits, 16-byte aligned or not, with `k` reported tokens on a device of
 * `cus` compute units: slices a row and tokens a slice.  No device work. */
lsamp_status lsamp_test_plan_rank(int32_t rows, int32_t vocab, int32_t dtype, int32_t k,
                                  int32_t lse, int32_t aligned, int32_t cus, int32_t* slices,
                                  int32_t* slice_len);

/* For each of the first `rows` rows of the context's last sampling or
 * verification launch (not the top-k kernel's): 1 when the row was drawn from
 * its slices' lists, 0 when it took the histogram path.  Synchronous. */
lsamp_status lsamp_test_rows_from_lists(lsamp_context* ctx, int32_t rows, int32_t* out);

#ifdef __cplusplus
}
#endif

#endif /* LSAMP_TESTING_H */
