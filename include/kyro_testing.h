/*
 * kyro_testing.h — test-only controls of libkyro_verify. No counterpart in the reference: these
 * exist so that the library's own tests can force conditions a correct caller never produces.
 * A production caller never calls them; a process that does not call them behaves exactly as
 * if they did not exist (no environment variable or other implicit input is read).
 */
#ifndef KYRO_TESTING_H
#define KYRO_TESTING_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Caps the partial-state slots a balanced-schedule kyro_paged_attention_mq call sizes at `cap`
 * (process-wide; 0, the initial state, sizes the full bound). With a cap below what the plan
 * needs, the device plan latches an error and runs no item, and the next kyro_sync returns
 * KYRO_EINVAL. Returns the previous cap. */
int64_t kyro_testing_set_plan_slot_cap(int64_t cap);

struct kyro_paged_attention_params;

/* Tiles of a part that the many-row attention kernel gives the row groups of a sequence of `ctx` tokens in a
 * call of these params (256 CUs), and the most parts of one in *splits; 0 where the kernel lists its work
 * on the device, negative where the call does not take that kernel. No device call. */
int kyro_testing_prefill_part_tiles(const struct kyro_paged_attention_params* params, int has_q_start_loc,
                                    int64_t ctx, int* splits);

#ifdef __cplusplus
}
#endif

#endif /* KYRO_TESTING_H */
