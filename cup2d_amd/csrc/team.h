// team.h -- the on-chip solve: one kernel runs whole FP64 BiCGSTAB solves
// with the vectors held in registers (team.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <vector>

#include "../../include/cup2d_chip.h"
#include "kernels.h"

namespace cup2d {

// One solve of a launch: blocks b0 .. b0 + nb - 1 of the operator, taken by a
// team of nwg workgroups of bpw consecutive blocks each (the last one fewer).
struct TeamTask {
  int b0, nb;
  int nwg, bpw;
  int ticket0;        // first ticket of the team: workgroup `rank` holds ticket0 + rank
  int slot0;          // first of the team's exchange words, in units of TEAM_SLOT_WORDS
  int e0, e1;         // explicit rows (ELL slots) of these blocks
  int mean_row;       // replaced row, or -1
  int order;          // tasks before this one
};

constexpr int TEAM_MAX_WG = 256;        // workgroups of a team: at most one per CU
constexpr int TEAM_MAX_BLOCKS = 64 * TEAM_MAX_WG;  // largest mesh solved on chip
constexpr int TEAM_PHASES = 5;          // cup2d_ps_phase

// Words of the exchange area per workgroup slot (see team.hip).
constexpr int TEAM_NQ = 4;              // quantities of one exchange
constexpr int TEAM_SLOT_WORDS = 2 * 2 * TEAM_NQ;
// Copies of the exchange words, each read by some of the workgroups: one up to
// 64 workgroups, then one per 32 (a line that 250 workgroups poll is slow to
// reach).  Sums by groups of 16 and then over the groups, two waits with 16
// values each, took 1-2 us an iteration more on 96-256 workgroups.
__host__ __device__ constexpr int team_copies(int nwg) { return nwg <= 64 ? 1 : (nwg + 31) / 32; }
// Exchange words of a team.
constexpr size_t team_words(int nwg) { return (size_t)nwg * TEAM_SLOT_WORDS * team_copies(nwg); }

// Places (words) in a task's part of a halo buffer, block b counted from the
// task's first: the faces of every block (8 cells each, Xm, Xp, Ym, Yp), then
// every block whole; 64 bytes that one workgroup writes and another reads lie
// together.  Counted over a whole batch they would leave 32 bits from 22 million
// blocks (of 33) on.
constexpr int HALO_BLOCK = 96;
__host__ __device__ constexpr int halo_face(int b, int f) { return 32 * b + 8 * f; }
__host__ __device__ constexpr int halo_cell(int nb, int b) { return 32 * nb + 64 * b; }
static_assert(halo_cell(TEAM_MAX_BLOCKS, TEAM_MAX_BLOCKS - 1) + 63 == (long long)HALO_BLOCK * TEAM_MAX_BLOCKS - 1 &&
                  halo_face(TEAM_MAX_BLOCKS - 1, 3) + 7 == halo_cell(TEAM_MAX_BLOCKS, 0) - 1,
              "places of the largest task");

struct TeamArgs {
  OpView A;
  const int2 *fid;
  const double *pc;                     // FP64 MFMA fragments of P_inv's classes
  const double *b, *x0;
  double *out;
  double *halo;                         // [3 n] what the workgroups read of each other (two buffers)
  double *xopt;                         // [n] work vector
  int n_codes;                          // entries of A.etab
  const TeamTask *task;                 // [n_tasks], or null: the one task `one`
  TeamTask one;
  int n_tasks, n_tickets;
  int start;                            // TeamStart
  int mean_rows, norm_max;              // a mean row among the tasks, the infinity norm
  int form_polls;                       // polls before the wait for a team to form fails, earlier tasks ended
  Scal *st;                             // [n_tasks] marker state in, final state out
  unsigned long long *slots;            // exchange words of all teams, zero at launch
  int *ctl;                             // {next ticket, failure, ended tasks}, zero at launch
  unsigned long long *phase;            // [n_tasks][TEAM_PHASES] ticks of 10 ns, or null
};

// What the start of a solve (and of a residual replacement) also decides.
enum TeamStart {
  TEAM_PLAIN = 0,     // nothing (the FP64 single solve: evaluate alone)
  TEAM_CHECKED = 1,   // a non-finite residual ends the solve, a zero one is convergence
  TEAM_ACCEPTS = 2,   // ... and a start within the tolerance is convergence too
  TEAM_REFINES = 3,   // ... and the solve is a sequence of passes (iterative refinement): max_restarts
                      // holds for each, and whatever ends one -- the recurrence's claim, its restarts, the
                      // iteration cap -- is followed by the residual of the best iterate
};

// Blocks per workgroup of a launch shape.
enum TeamShape { TEAM_16 = 0, TEAM_32 = 1, TEAM_48 = 2, TEAM_64 = 3, TEAM_SHAPES = 4 };
inline int team_blocks(int shape) { return shape == TEAM_64 ? 64 : 16 * (shape + 1); }

// Polls before a wait inside a team fails: 0.15 us each on 8 workgroups, 0.23 on
// 192, 0.3-0.5 s in all.
constexpr int TEAM_POLLS = 1 << 21;

// Workgroups of a shape that this device runs at once (0: unknown; the
// kernels' LDS size is allowed here, so a shape is asked for before its launch).
int team_resident(int shape);

// What a handle's cup2d_ps_set_on_chip says, and what came of its last solves.
struct TeamUse {
  int mode = CUP2D_PS_CHIP_AUTO;
  int polls = TEAM_POLLS;   // for a team to form
  bool ran = false;         // the last solve, on chip
  int wait = 0, next = 1;   // solves until the chip is tried again, and after the next failure

  // Whether to try the chip for this solve.  After a launch that could not run
  // (the runtime refuses cooperative launches while another process makes them,
  // which takes 0.5 ms; a wait that ends at its limit takes 0.3-0.5 s) it is
  // left out for one solve, then for twice as many each time it fails again: the
  // cause may pass, and where it stays the attempts become few.
  bool now() {
    if (mode == CUP2D_PS_CHIP_OFF) return false;
    if (wait > 0) {
      wait--;
      return false;
    }
    return true;
  }
  void tried(bool done) {
    wait = done ? 0 : next;
    next = done ? 1 : next < 1024 ? 2 * next : next;
  }
  void new_mesh() { wait = 0, next = 1; }
};
inline bool team_use_set(TeamUse &u, int mode, int polls) {
  if (mode < CUP2D_PS_CHIP_AUTO || mode > CUP2D_PS_CHIP_SHORT || polls < 0) return false;
  u.mode = mode;
  u.polls = polls > 0 ? polls : TEAM_POLLS;
  return true;
}
// Workgroups to launch of a shape: `grid`, whose first team has nwg, or what the
// mode asks for in their place.
inline int team_grid(const TeamUse &u, int shape, int grid, int nwg) {
  return u.mode == CUP2D_PS_CHIP_REFUSED ? team_resident(shape) + 1
         : u.mode == CUP2D_PS_CHIP_SHORT && nwg > 1 ? nwg - 1 : grid;
}

// Splits nb blocks over a team of workgroups of at most `most` blocks.
inline void team_split(int nb, int most, TeamTask &t) {
  t.nb = nb;
  t.nwg = (nb + most - 1) / most;
  t.bpw = (nb + t.nwg - 1) / t.nwg;
  t.nwg = (nb + t.bpw - 1) / t.bpw;
}

// The fragments of P_inv (make_pfrag64, make_pclass64, make_pfrag) in one new
// buffer on the device, in this order; nothing is left of it where that fails.
inline hipError_t upload_pinv(const std::vector<double> &f64, const std::vector<double> &c64,
                              const std::vector<uint16_t> &f16, double *&out) {
  std::vector<double> all(f64);
  all.insert(all.end(), c64.begin(), c64.end());
  const size_t n = all.size(), bytes = n * sizeof(double) + f16.size() * sizeof(uint16_t);
  all.resize((bytes + sizeof(double) - 1) / sizeof(double));
  std::memcpy(all.data() + n, f16.data(), f16.size() * sizeof(uint16_t));
  double *d = nullptr;
  hipError_t e = hipMalloc((void **)&d, bytes);
  if (e == hipSuccess) e = hipMemcpy(d, all.data(), bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) out = d;
  else if (d) (void)hipFree(d);
  return e;
}

// Launches the solves on `stream` with `grid` workgroups, no more than
// team_resident and no fewer than any task's team (the exchange words and ctl
// are cleared first).  Nothing is allocated.
hipError_t team_launch(const TeamArgs &a, int shape, size_t n_words, int grid, hipStream_t stream);

}  // namespace cup2d
