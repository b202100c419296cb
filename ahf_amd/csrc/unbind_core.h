/*
 * unbind_core.h -- rules of the unbinding kernels that the host replays as
 * well (tests/emu/handup_check.c).
 */
#ifndef AHF_UNBIND_CORE_H
#define AHF_UNBIND_CORE_H

#include <stdint.h>

#ifdef __HIPCC__
#define AHF_HD __host__ __device__ inline
#else
#define AHF_HD static inline
#endif

/*
 * The register form's hand-up (unbind_resident): whether a thread's statuses
 * changed in a round, so that the wavefronts above its own have to take the
 * totals again.  Wavefront w's statuses follow from the totals below it
 * alone, so wavefront 0 changes in round 1 at most, w in round w + 1 at most,
 * and the rounds end by the number of wavefronts plus one, whatever the
 * velocities are.  The totals themselves would not do: a NaN velocity stays
 * bound (rem_unbound removes a member only if its speed exceeds the limit),
 * and a NaN total differs from itself.
 */
AHF_HD int ahf_handup_moved(uint32_t before, uint32_t now) { return before != now; }

#endif /* AHF_UNBIND_CORE_H */
