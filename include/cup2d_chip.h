/* Where the solves of a handle of cup2d_poisson.h run.
 *
 * A mesh of at most 16,384 blocks is solved on chip: by one launch of as many
 * workgroups as it takes, which are on the device at once and wait for each
 * other.  So is a batch whose meshes all are (with mean_constraint 0).  Larger
 * meshes, the unfused comparator, and a solve whose launch on chip could not run
 * are solved by launches per kernel.  No counterpart in the reference. */
#ifndef CUP2D_CHIP_H
#define CUP2D_CHIP_H

#include "cup2d_poisson.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The last two modes are for tests of the hand-over between the two paths. */
typedef enum {
  CUP2D_PS_CHIP_AUTO = 0,    /* on chip where the mesh fits (default) */
  CUP2D_PS_CHIP_OFF = 1,     /* by launches per kernel */
  CUP2D_PS_CHIP_REFUSED = 2, /* more workgroups are asked for than fit, which the runtime refuses */
  CUP2D_PS_CHIP_SHORT = 3    /* one workgroup fewer than the solve takes (if it takes two or more):
                                the others' wait for it ends at its limit */
} cup2d_ps_chip;

/* Sets the mode of a handle's solves from now on.  form_polls: polls (0.15-0.25 us
 * each) a workgroup waits for the others to be there, once the instances of a batch
 * before its own have ended; 0 = the default, 2^21. */
int cup2d_ps_set_on_chip(cup2d_ps *h, int mode, int form_polls);
int cup2d_psb_set_on_chip(cup2d_psb *h, int mode, int form_polls);

/* Whether the handle's last solve ran on chip. */
int cup2d_ps_on_chip(const cup2d_ps *h);
int cup2d_psb_on_chip(const cup2d_psb *h);

#ifdef __cplusplus
}
#endif

#endif /* CUP2D_CHIP_H */
