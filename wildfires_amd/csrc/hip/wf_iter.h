/*
 * wf_iter.h -- the convergence flag of the pressure iteration (WfIterCtl::done)
 * and who returns on it.  Host/device-neutral: the CPU check runs these rules.
 *
 * The check of solve m is one workgroup of solve m + 1's first pass, so that
 * pass's other workgroups read the flag while it may be written, each
 * wavefront for itself.  They have barriers, and fill LDS that the wavefronts
 * share, so all wavefronts of a workgroup have to decide alike whichever value
 * they see.  The flag therefore holds the number of the solve that ended the
 * iteration (its index plus 1; 0: none yet), and a first pass that checks solve
 * `check` returns only for an earlier one: 0 and check + 1, the two values it
 * can see while its own check writes, both mean that it goes on.  If solve
 * `check` ended the iteration, the pass has written what nothing reads any more;
 * every later pass, for which the flag no longer changes, returns at once.
 */
#ifndef WF_ITER_H
#define WF_ITER_H

#if defined(__HIPCC__)
#define WF_ITER_HD __host__ __device__ static __forceinline__
#else
#define WF_ITER_HD static inline
#endif

/* the flag after the check of solve m */
WF_ITER_HD int wf_iter_flag(int ended, int m) { return ended ? m + 1 : 0; }
/* whether a first pass that checks solve `check` (-1: none) returns at once */
WF_ITER_HD int wf_first_pass_returns(int flag, int check) { return flag != 0 && (check < 0 || flag <= check); }
/* whether a later pass of a solve, or a check, returns at once */
WF_ITER_HD int wf_pass_returns(int flag) { return flag != 0; }

#endif
