// team.hip -- whole FP64 BiCGSTAB solves in one kernel.
//
// The iteration of BiCGSTAB.cu:412-620 (restart, best iterate, stopping
// norms) with the vectors r, rhat, p, nu, z, t and x of a workgroup's blocks in
// its registers for the whole solve.  A team of co-resident workgroups
// advances one mesh; the only data that leave a workgroup are the cells of
// z = P v that another workgroup's rows read (the operator's halo) and the
// partial sums of the dot products.
//
// What bounds it: an iteration has four points where the workgroups wait for
// each other (z's halo twice, (rhat, nu) with the size of the r before, and
// omega's sums with those of the next rho), each one store and one load past
// the L2s, which are not coherent between the XCDs: 0.7-1 us for a halo, 1.0 us
// (8 workgroups) to 2-3 us (250) for sums.  A fence that writes an L2 back
// costs more than a kernel boundary; here every shared word is written and
// read by relaxed agent-scope accesses, and a waiting workgroup polls the data
// themselves: partial sums carry the exchange's number in the upper half of
// each word, and a halo word holds a NaN that no arithmetic returns until its
// value arrives.  Between the waits a wave's instructions count (one to three
// waves per SIMD), above all the taken branches and the chains of LDS reads:
// the two halves of an iteration are one straight line (as one body with the
// mode as a variable they took 10.6 us on 128 blocks, 8.0 so), everything an
// explicit row needs lies in LDS, and the addresses of a thread's halo words
// in registers.  What is the same in every lane is kept in scalar registers
// (uni): in vector ones the vectors were spilled to memory (64 blocks per
// workgroup: 20.5 us on 16,384 blocks, 17.6 without).  There are too many of
// them: 129-184 scalar registers are spilled to lanes of vector ones, whose
// reloads lie in the loop, and 8-24 bytes a lane of flags to memory; of the
// vectors the 48-block shape spills 2 registers (12 with the infinity norm).
//
// Measured (us per iteration to a relative residual of 1e-12, against five
// kernels per iteration replayed from a graph): 128 blocks 7.7 against 24.0,
// 1448 blocks 10.5 against 27.9, 8348 blocks 15.4 against 49.9, 16,229 blocks
// 18.8 against 64.8.  One workgroup of 64 blocks alone takes 7.4 us, of 16 4.3 us:
// the rest is the waits and the slowest of the workgroups.
//
// Teams form by tickets: a workgroup takes the next ticket, which names its
// task and its rank, and when its task is solved takes another.  Tickets are
// taken in order by running workgroups, so the lowest unfinished task always
// has or gets its whole team (a cooperative launch: no more workgroups than
// fit) and every wait ends; a wait beyond its limit marks the launch as
// failed and every workgroup leaves.  Workgroups that wait for a team to form
// wait for earlier tasks, however long those run; their limit is for a launch
// that did not get its workgroups.

#include "team.h"

#include <atomic>

namespace cup2d {
namespace {

typedef unsigned long long u64;

constexpr int ZS = 66;                    // LDS row of a block: 16-byte aligned, 16 blocks over all banks
constexpr int TEAM_MAX_CONFIRM = 64;      // residual confirmations of a mixed solve

__device__ __forceinline__ u64 ld_agent(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(u64 *p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// N pairs of words (16 bytes each, past the caches), the wait included.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void ld_pairs(const u64 *const (&p)[1], u32x4 (&v)[1]) {
  asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v[0]) : "v"(p[0]) : "memory");
}
__device__ __forceinline__ void ld_pairs(const u64 *const (&p)[2], u32x4 (&v)[2]) {
  asm volatile(
      "global_load_dwordx4 %0, %2, off sc1\n\tglobal_load_dwordx4 %1, %3, off sc1\n\ts_waitcnt vmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1])
      : "v"(p[0]), "v"(p[1])
      : "memory");
}
__device__ __forceinline__ void ld_pairs(const u64 *const (&p)[4], u32x4 (&v)[4]) {
  asm volatile(
      "global_load_dwordx4 %0, %4, off sc1\n\tglobal_load_dwordx4 %1, %5, off sc1\n\t"
      "global_load_dwordx4 %2, %6, off sc1\n\tglobal_load_dwordx4 %3, %7, off sc1\n\ts_waitcnt vmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3])
      : "memory");
}

// A value that is the same in every lane, as the compiler sees it too: the
// branches on it then keep one copy of the registers either side updates.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = uni((int)b), hi = uni((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Wave reductions by DPP (row shifts, then row broadcasts; the total in lane
// 63): a step is two register moves and an add, where a shuffle through LDS
// takes its latency.  Lanes without a source add 0; the maxima are of
// absolute values, so 0 serves there too.
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <bool MAX>
__device__ __forceinline__ double dpp_total(double v) {
  auto op = [](double a, double b) { return MAX ? nmax(a, b) : a + b; };
  v = op(v, dpp<0x111>(v));  // row_shr 1, 2, 4, 8
  v = op(v, dpp<0x112>(v));
  v = op(v, dpp<0x114>(v));
  v = op(v, dpp<0x118>(v));
  v = op(v, dpp<0x142>(v));  // row_bcast 15, 31
  v = op(v, dpp<0x143>(v));
  return v;
}

// A word of z that has not arrived: a signalling NaN, which no arithmetic
// returns.
constexpr u64 EMPTY = 0x7ff4c2d0a11c0de5ull;

constexpr int face_rows(int blocks) { return blocks * 28; }  // a block has 28 cells on its faces
constexpr int ENT = 14, HALF = ENT / 2;                      // entries of an explicit row kept in LDS (13 occur)
constexpr int TAB = 256;                                     // coefficients kept in LDS

template <int WGS, int T>
struct Shared {
  static constexpr int BPW = WGS / 256 * T * TILE, NW = WGS / 64;
  static constexpr int GHOST0 = BPW * ZS, GHOSTS = BPW * 40;  // first, most cells of other workgroups
  static constexpr int ITEMS = BPW * 12;                      // a block's 4 faces and 8 rows
  // Explicit rows kept in LDS, and those of more than HALF entries among them
  // (a third of the rows; 300-625 and 100-280 occur on 64 blocks of small graded
  // meshes, a row beyond them is read from memory: 9 such meshes took 19.7 ms
  // when 512 rows were kept, 14.5 so, 32 of 400-1,600 blocks 29.2 and 17.4).
  static constexpr int ROWS = BPW == 64 ? 704 : BPW == 48 ? 768 : face_rows(BPW), WIDE = BPW == 64 ? 288 : ROWS;
  double z[GHOST0 + GHOSTS];        // the workgroup's blocks (product inputs, then z), then the ghosts
  double part[GHOST0];              // P v of the blocks, by class
  double ye[face_rows(BPW)];        // A z of the explicit rows
  double tab[TAB];
  double red[TEAM_NQ][NW], tot[TEAM_NQ];  // a wave per quantity: TEAM_NQ <= NW
  u64 mask[BPW];
  double h2[BPW];
  int4 face[BPW];                   // where z across each face lies (Xm, Xp, Ym, Yp); the block's own cells
                                    // where no plain neighbour does (a wall's term vanishes)
  int ghost[GHOSTS];                // where in the halo buffer each ghost comes
  unsigned ent[HALF][ROWS];         // entries of the explicit rows: LDS index, coefficient << 16
  unsigned wide[HALF][WIDE];        // those from HALF on
  int erow[face_rows(BPW)];         // place in `wide` of each explicit row in LDS, ELL slot of the others
  int eoff[BPW + 1];                // first explicit row of each block
  unsigned char ewid[face_rows(BPW)];  // entries, | 64 with ghosts among them, | 192 read from memory
  int2 item[ITEMS];                 // what other workgroups read, 8 cells each: {first LDS index | stride 8 (bit
                                    // 16), place in the halo buffer / 8}
  u64 tick, phase[TEAM_PHASES];     // of the profile: not in registers, which the loop needs
  int ng, ni, nf, nw, ticket, bad;  // ghosts, items, explicit rows with ghosts, wide ones
  int restarts;                     // of the passes before this one
};

// The running workgroup: what its functions share.
template <int WGS, int T>
struct Ctx {
  typedef Shared<WGS, T> S;
  const TeamArgs &a;
  S &s;
  int tid, lane, w, q, j, grp, c0;  // wave within its tile, MFMA column / k slot, first cell
  TeamTask t;
  int rank, b0, nb;                 // first block, blocks
  u64 *slots;
  double *halo0;                    // the task's part of the halo buffer
  int copies, copy, slab;           // copies of the exchange words, the one read here, words of a copy
  unsigned ep, zp;                  // number of the exchange, parity of z's buffer
  int ni8, ng, nf;                  // words that others read, ghosts, explicit rows with ghosts
  int iz, io, ig;                   // the thread's first such word (LDS index, place), its first ghost's place
  bool dead;

  __device__ __forceinline__ Ctx(const TeamArgs &aa, S &ss) : a(aa), s(ss), dead(false) { place(); }

  // The thread's place, computed anew: kept out of the compiler's sight, so
  // that the dozens of addresses that follow from it are recomputed where
  // they are used and don't hold registers through the loop (with T = 2 they
  // pushed the vectors out to memory).
  __device__ __forceinline__ void place() {
    tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    lane = tid & 63;
    q = lane >> 4;
    j = lane & 15;
    const int wv = uni(tid >> 6);
    w = wv & 3;
    grp = wv >> 2;
    c0 = 16 * w + 4 * q;
  }

  __device__ __forceinline__ int lb(int tt) const { return (grp * T + tt) * TILE + j; }
  __device__ __forceinline__ bool ok(int tt) const { return lb(tt) < nb; }
  __device__ __forceinline__ long cell(int tt) const { return (long)(b0 + (ok(tt) ? lb(tt) : 0)) * 64 + c0; }
  // the task's halo buffer of this z (halo_face, halo_cell)
  __device__ __forceinline__ double *halo() const { return halo0 + (zp ? (long)HALO_BLOCK * a.A.nb : 0); }

  // every 1024 polls: whether to give up (the launch failed, or the limit; a
  // negative one is that of the wait for the team to form, which counts from the
  // end of the tasks before it: their workgroups are the ones awaited)
  __device__ __forceinline__ bool give_up(int &n, int limit) {
    if (((++n) & 1023) != 0) return false;
    if (limit < 0) {
      limit = -limit;
      if (__hip_atomic_load(a.ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < t.order) n = 0;
    }
    if (n < limit && !__hip_atomic_load(a.ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    __hip_atomic_store(a.ctl + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s.bad = 1;
    return true;
  }

  // z at a cell of another workgroup, once it has arrived; v: a first look
  __device__ __forceinline__ double remote(const double *p, u64 v, int limit) {
    const u64 *w64 = reinterpret_cast<const u64 *>(p);
    int n = 0;
    while (v == EMPTY && !dead && !give_up(n, limit)) v = ld_agent(w64);
    return __longlong_as_double((long long)v);
  }

  // The cells that others read go to the halo buffer (from LDS), or are
  // emptied there.
  template <bool EMPTIES>
  __device__ __forceinline__ void publish(double *buf) {
    if (tid < ni8)
      st_agent(reinterpret_cast<u64 *>(buf + io), EMPTIES ? EMPTY : (u64)__double_as_longlong(s.z[iz]));
#pragma unroll 1
    for (int i = tid + WGS; i < ni8; i += WGS) {
      int at, to;
      word(i, at, to);
      st_agent(reinterpret_cast<u64 *>(buf + to), EMPTIES ? EMPTY : (u64)__double_as_longlong(s.z[at]));
    }
  }
  // word i of those that others read: its LDS index and its place in the halo buffer
  __device__ __forceinline__ void word(int i, int &at, int &to) const {
    const int2 it = s.item[i >> 3];
    at = (it.x & 0xffff) + (it.x >> 16 ? 8 * (i & 7) : i & 7);
    to = 8 * it.y + (i & 7);
  }

  // After the pass's last exchange everyone has read its z: the words are
  // emptied (that is complete before the next exchange, which lies before
  // their next use) and the other buffer is next.
  __device__ __forceinline__ void clear() {
    publish<true>(halo());
    zp ^= 1;
  }

  // The total of the n values at p, once they have come, 64 NS or fewer.
  template <int NS, bool MAXLAST>
  __device__ __forceinline__ double gather(const u64 *p, int n, bool mx, int limit) {
    auto op = [mx](double x, double y) { return MAXLAST && mx ? nmax(x, y) : x + y; };
    const u64 *at[NS];
    u32x4 v[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) at[i] = p + 2 * min(i * 64 + lane, n - 1);
    unsigned off;
    int polls = 0;
    do {
      ld_pairs(at, v);
      off = 0;
#pragma unroll
      for (int i = 0; i < NS; i++) off |= (v[i].y ^ ep) | (v[i].w ^ ep);
    } while (off && !dead && !give_up(polls, limit));
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < NS; i++)
      r = op(r, i * 64 + lane < n ? __longlong_as_double((long long)v[i].z << 32 | v[i].x) : 0.0);
    r = MAXLAST && mx ? dpp_total<true>(r) : dpp_total<false>(r);
    const long long b = __double_as_longlong(r);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
  }

  // Sums (the last one a maximum with MAXLAST) of the NQ quantities over
  // the team, in a fixed order, so that every workgroup holds the same totals:
  // lanes, waves, ranks.  The totals are in s.tot.  A wave per quantity
  // publishes the workgroup's sum and gathers the team's.
  template <int NQ, bool MAXLAST>
  __device__ __forceinline__ void exchange(double (&v)[NQ], int limit) {
    const int wv = uni(tid >> 6);
#pragma unroll
    for (int k = 0; k < NQ; k++)
      v[k] = MAXLAST && k == NQ - 1 ? dpp_total<true>(v[k]) : dpp_total<false>(v[k]);
    if (lane == 63)
#pragma unroll
      for (int k = 0; k < NQ; k++) s.red[k][wv] = v[k];
    // what this workgroup emptied is empty before it says that it is here
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    ep++;
    if (wv < NQ) {
      const bool mx = MAXLAST && wv == NQ - 1;
      auto op = [mx](double x, double y) { return MAXLAST && mx ? nmax(x, y) : x + y; };
      const double2 *rp = reinterpret_cast<const double2 *>(s.red[wv]);
      double r = 0.0;
#pragma unroll
      for (int i = 0; i < S::NW / 2; i++) {
        const double2 u = rp[i];
        r = op(op(r, u.x), u.y);
      }
      const int n = t.nwg;
      if (n > 1) {
        u64 *base = slots + (ep & 1 ? slab * copies : 0) + 2 * wv * n;
        // a value is two words that carry the exchange's number
        const u64 b = (u64)__double_as_longlong(r), tag = (u64)ep << 32;
        if (lane < 2 * copies)
          st_agent(base + (lane >> 1) * slab + 2 * rank + (lane & 1), tag | (lane & 1 ? b >> 32 : b & 0xffffffffull));
        const u64 *mine = base + copy * slab;
        r = n <= 64 ? gather<1, MAXLAST>(mine, n, mx, limit)
            : n <= 128 ? gather<2, MAXLAST>(mine, n, mx, limit) : gather<4, MAXLAST>(mine, n, mx, limit);
      }
      if (lane == 0) s.tot[wv] = r;
    }
    __syncthreads();
    dead = dead || uni(s.bad) != 0;
  }

  __device__ __forceinline__ void to_lds(const double (&z)[T][4]) {
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
      double2 *d = reinterpret_cast<double2 *>(s.z + lb(tt) * ZS + c0);
      d[0] = make_double2(z[tt][0], z[tt][1]);
      d[1] = make_double2(z[tt][2], z[tt][3]);
    }
  }
  __device__ __forceinline__ void from_lds(int i, double (&v)[4]) const {
    const double2 *d = reinterpret_cast<const double2 *>(s.z + i);
    const double2 u0 = d[0], u1 = d[1];
    v[0] = u0.x; v[1] = u0.y; v[2] = u1.x; v[3] = u1.y;
  }

  // z = P z of the thread's cells, by parts that are even or odd in x and y
  // (make_pclass64): the tile's wave w forms the quadrant of part w, 4
  // products in place of 16, and the parts are put together through LDS.
  // An iteration of 16,384 blocks took 17.6 us with the 64 x 64 product (and its
  // operands in 32 KB of LDS), 16.8 so; of 8348 graded blocks 16.4 and 15.2; the
  // 64-instance batch 361 ms and 300 ms.
  __device__ __forceinline__ void prec(const double (&F)[4], double (&z)[T][4]) {
    to_lds(z);
    __syncthreads();
    const double sx = w & 1 ? -1.0 : 1.0, sy = w & 2 ? -1.0 : 1.0;
    f64x4 acc[T];
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
      double lo[2][4], hi[2][4], in[4];  // rows q and 7 - q
      from_lds(lb(tt) * ZS + 8 * q, lo[0]);
      from_lds(lb(tt) * ZS + 8 * q + 4, lo[1]);
      from_lds(lb(tt) * ZS + 8 * (7 - q), hi[0]);
      from_lds(lb(tt) * ZS + 8 * (7 - q) + 4, hi[1]);
#pragma unroll
      for (int k = 0; k < 4; k++)
        in[k] = fma(sy, fma(sx, hi[1][3 - k], hi[0][k]), fma(sx, lo[1][3 - k], lo[0][k]));
      acc[tt] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 4; k++) acc[tt] = __builtin_amdgcn_mfma_f64_16x16x4f64(F[k], in[k], acc[tt], 0, 0, 0);
    }
    if constexpr (T == 1) settle(acc[0]);
    else settle(acc[0], acc[T - 1]);
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
      double2 *d = reinterpret_cast<double2 *>(s.part + lb(tt) * ZS + c0);
      d[0] = make_double2(acc[tt][0], acc[tt][1]);
      d[1] = make_double2(acc[tt][2], acc[tt][3]);
    }
    __syncthreads();
    const int row = 2 * w + (q >> 1), yq = row < 4 ? row : 7 - row;
    const bool right = q & 1;  // the row's right half: the quadrant's mirror image
    const double s2 = w < 2 ? 1.0 : -1.0, s1 = right ? -1.0 : 1.0;
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
      double v[4][4];
#pragma unroll
      for (int cl = 0; cl < 4; cl++) {
        const double2 *d = reinterpret_cast<const double2 *>(s.part + lb(tt) * ZS + 16 * cl + 4 * yq);
        const double2 u0 = d[0], u1 = d[1];
        v[cl][0] = u0.x; v[cl][1] = u0.y; v[cl][2] = u1.x; v[cl][3] = u1.y;
      }
      double o[4];
#pragma unroll
      for (int k = 0; k < 4; k++) o[k] = fma(s1, fma(s2, v[3][k], v[1][k]), fma(s2, v[2][k], v[0][k]));
#pragma unroll
      for (int k = 0; k < 4; k++) z[tt][k] = right ? o[3 - k] : o[k];
    }
  }

  // ye = A z of the explicit rows whose kind (0: all entries in LDS from the
  // start, 64: some are ghosts, or the row is read from memory) is this: a
  // thread per row.
  __device__ __forceinline__ void explicit_rows(int kind, const double *zb, int limit) {
    const int ne = uni(s.eoff[nb]);
    for (int k = tid; k < ne; k += WGS) {
      const int how = s.ewid[k], width = how & 63;
      if ((how & 64) != kind) continue;
      double sum = 0.0;
      if (how < 128) {
        auto add = [&](const unsigned *from, int stride) __attribute__((always_inline)) {
          unsigned en[HALF];
#pragma unroll
          for (int i = 0; i < HALF; i++) en[i] = from[i * stride];
#pragma unroll
          for (int i = 0; i < HALF; i++) sum += s.tab[en[i] >> 16] * s.z[en[i] & 0xffffu];
        };
        add(s.ent[0] + k, S::ROWS);
        if (width > HALF) add(s.wide[0] + s.erow[k], S::WIDE);
      } else {
        const int e = s.erow[k];
        for (int i = 0; i < width; i++) {
          const long at = (long)i * a.A.n_exc + e;
          const int col = a.A.ecol[at], l = (col >> 6) - b0;
          const double v =
              (l >= 0 && l < nb) ? s.z[l * ZS + (col & 63)] : remote(zb + place_of(a.A.erow[e] >> 6, col), EMPTY, limit);
          sum += a.A.etab[a.A.ecode[at]] * v;
        }
      }
      s.ye[k] = sum;
    }
  }

  // y = A z of the thread's cells (0 past the last block, where z is 0)
  __device__ __forceinline__ void spmv(const double (&z)[T][4], double (&y)[T][4], int limit) {
    const double *zb = halo();
    to_lds(z);
    int4 face[T];
    u64 mask[T];
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
      face[tt] = s.face[lb(tt)];
      mask[tt] = s.mask[lb(tt)];
    }
    __syncthreads();
    publish<false>(halo());
    // The ghosts are asked for, the explicit rows without any are computed
    // while they travel, and the others follow.
    u64 v0 = 0;
    if (tid < ng) v0 = ld_agent(reinterpret_cast<const u64 *>(zb + ig));
    explicit_rows(0, zb, limit);
    if (tid < ng) {
      s.z[S::GHOST0 + tid] = remote(zb + ig, v0, limit);
#pragma unroll 1
      for (int g = tid + WGS; g < ng; g += WGS) s.z[S::GHOST0 + g] = remote(zb + s.ghost[g], EMPTY, limit);
    }
    __syncthreads();
    if (nf > 0) {
      explicit_rows(64, zb, limit);
      __syncthreads();
    }
    const int row = 2 * w + (q >> 1), ix0 = 4 * (q & 1);
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
      const int base = lb(tt) * ZS;
      const int4 f = face[tt];
      const int fx = ix0 == 0 ? f.x : f.y;
      const double mid = s.z[base + row * 8 + (ix0 == 0 ? 4 : 3)];  // across the middle of the row
      const double hx = s.z[fx + (fx < S::GHOST0 ? 8 * row : row)];
      double dn[4], up[4];
      from_lds((row > 0 ? base + (row - 1) * 8 : f.z) + ix0, dn);
      from_lds((row < 7 ? base + (row + 1) * 8 : f.w) + ix0, up);
      const double lo = ix0 == 0 ? hx : mid, hi = ix0 == 0 ? mid : hx;
#pragma unroll
      for (int k = 0; k < 4; k++) {  // face order Ym, Xm, Xp, Yp as the other operator kernels
        const double xl = k > 0 ? z[tt][k > 0 ? k - 1 : 0] : lo;
        const double xr = k < 3 ? z[tt][k < 3 ? k + 1 : 3] : hi;
        y[tt][k] = ((dn[k] + xl) + xr) + up[k] - 4.0 * z[tt][k];
      }
      const u64 m = mask[tt];
      const unsigned em = (unsigned)(m >> c0) & 15u;
      if (em) {  // the block's explicit rows come in the order of its mask's bits
        int at = s.eoff[lb(tt)] + __popcll(m & ((1ull << c0) - 1));
#pragma unroll
        for (int k = 0; k < 4; k++)
          if ((em >> k) & 1u) y[tt][k] = s.ye[at++];
      }
    }
  }

  // Where in the halo buffer a cell of another workgroup comes, for a row of
  // block b: with the face that a same-level neighbour shows b (the only
  // cells of it that b's rows read), or with the whole block.
  __device__ __forceinline__ int place_of(int b, int col) const {
    const int4 n4 = a.A.nbr[b];
    const int blk = col >> 6, ix = col & 7, iy = (col >> 3) & 7;
    if (n4.x == blk && ix == 7) return halo_face(blk - t.b0, 1) + iy;
    if (n4.y == blk && ix == 0) return halo_face(blk - t.b0, 0) + iy;
    if (n4.z == blk && iy == 7) return halo_face(blk - t.b0, 3) + ix;
    if (n4.w == blk && iy == 0) return halo_face(blk - t.b0, 2) + ix;
    return halo_cell(t.nb, blk - t.b0) + (col & 63);
  }

  // Headers, ghosts and explicit rows of the workgroup's blocks.
  __device__ __forceinline__ void lay_out() {
    if (tid == 0) s.ng = s.ni = s.nf = s.nw = s.restarts = 0;
    __syncthreads();
    // LDS index of 8 cells of another workgroup, from `first` of the halo buffer on
    auto ghosts = [&](int first) -> int {
      const int g = atomicAdd(&s.ng, 8);
#pragma unroll 1
      for (int i = 0; i < 8; i++) s.ghost[g + i] = first + i;
      return S::GHOST0 + g;
    };
#pragma unroll 1
    for (int l = tid; l < S::BPW; l += WGS) {
      const bool in = l < nb;
      const int b = b0 + (in ? l : 0);
      const int4 n4 = a.A.nbr[b];
      s.mask[l] = in ? a.A.mask[b] : 0ull;
      s.h2[l] = in ? a.A.h2[b] : 0.0;
      int at[4];
      bool whole = false;
      auto offer = [&](int base, bool column, int to) {
        s.item[atomicAdd(&s.ni, 1)] = make_int2(l * ZS + base | (column ? 1 << 16 : 0), to / 8);
      };
#pragma unroll 1
      for (int f = 0; f < 4; f++) {
        const int nv = f == 0 ? n4.x : f == 1 ? n4.y : f == 2 ? n4.z : n4.w;
        at[f] = l * ZS + (f == 1 ? 7 : f == 3 ? 56 : 0);
        if (!in) continue;
        if (nv >= 0) {
          if (nv >= b0 && nv < b0 + nb) {
            at[f] = (nv - b0) * ZS + (f == 0 ? 7 : f == 2 ? 56 : 0);  // the neighbour's facing row
          } else {
            at[f] = ghosts(halo_face(nv - t.b0, f ^ 1));
            offer(f == 1 ? 7 : f == 3 ? 56 : 0, f < 2, halo_face(b - t.b0, f));
          }
        } else if (nv == -2) {
          const int2 fd = a.fid[4 * (long)b + f];
          // the rows beside a coarse-fine face read up to three cells deep
          whole = whole || fd.x < b0 || fd.x >= b0 + nb || (fd.y >= 0 && (fd.y < b0 || fd.y >= b0 + nb));
        }
      }
      if (whole)
#pragma unroll 1
        for (int i = 0; i < 8; i++) offer(8 * i, false, halo_cell(t.nb, b - t.b0) + 8 * i);
      s.face[l] = make_int4(at[0], at[1], at[2], at[3]);
    }
    __syncthreads();
    if (tid == 0) {
      int n = 0;
#pragma unroll 1
      for (int l = 0; l <= S::BPW; l++) {
        s.eoff[l] = n;
        if (l < S::BPW) n += __popcll(s.mask[l]);
      }
    }
    __syncthreads();
#pragma unroll 1
    for (int e = t.e0 + tid; e < t.e1; e += WGS) {
      const int row = a.A.erow[e], l = (row >> 6) - b0;
      if (l < 0 || l >= nb) continue;
      const int k = s.eoff[l] + __popcll(s.mask[l] & ((1ull << (row & 63)) - 1));
      int width = 0, slot = 0;
      bool fits = k < S::ROWS && a.A.ell_w <= ENT, far = false;
#pragma unroll 1
      for (int i = 0; i < a.A.ell_w; i++) {
        const long at = (long)i * a.A.n_exc + e;
        const unsigned code = a.A.ecode[at];
        if (code) width = i + 1;
        fits = fits && code < TAB;
      }
      if (fits && width > HALF) {
        slot = atomicAdd(&s.nw, 1);
        fits = slot < S::WIDE;
      }
#pragma unroll 1
      for (int i = 0; i < (width > HALF ? ENT : HALF) && fits; i++) {  // entries past the row's end: 0.0 times its own value
        const long at = (long)i * a.A.n_exc + e;
        const unsigned code = i < width ? a.A.ecode[at] : 0;
        const int col = i < width ? a.A.ecol[at] : row, lc = (col >> 6) - b0;
        unsigned idx;
        if (lc >= 0 && lc < nb) {
          idx = lc * ZS + (col & 63);
        } else {
          const int g = atomicAdd(&s.ng, 1);
          far = true;
          fits = g < S::GHOSTS;
          if (fits) s.ghost[g] = place_of(row >> 6, col);
          idx = S::GHOST0 + g;
        }
        if (fits) (i < HALF ? s.ent[i][k] : s.wide[i - HALF][slot]) = idx | code << 16;
      }
      s.erow[k] = fits ? slot : e;
      if (far || !fits) atomicAdd(&s.nf, 1);
      s.ewid[k] = (unsigned char)(fits ? (far ? 64 : 0) + width : 192 + width);
    }
    __syncthreads();
    ni8 = 8 * uni(s.ni);
    ng = min(uni(s.ng), S::GHOSTS);
    nf = uni(s.nf);
    iz = io = 0;
    if (tid < ni8) word(tid, iz, io);
    ig = s.ghost[min(tid, max(ng - 1, 0))];
  }
};

#define CELLS                             \
  _Pragma("unroll") for (int tt = 0; tt < T; tt++) _Pragma("unroll") for (int k = 0; k < 4; k++)

// What a task may ask for: the 2-norm on the operator's plain form, the
// infinity norm on it, or the mean row with either.
enum { PLAIN, NORM_MAX, MEAN_ROW, KINDS };

// Two waves' worth of registers at least are left to each wave (256): with
// more, the compiler keeps products in the accumulation registers.
template <int WGS, int T, int KIND>
__global__ __launch_bounds__(WGS, WGS > 512 ? WGS / 256 : 2) void k_team(TeamArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef Shared<WGS, T> S;
  static_assert(sizeof(S) <= 160 * 1024, "LDS of a CU");
  static_assert(S::GHOST0 + S::GHOSTS <= 65536 && S::GHOSTS >= S::BPW * 32, "LDS indices");
  S &s = *reinterpret_cast<S *>(smem);
  Ctx<WGS, T> c(a, s);
  const int &tid = c.tid;
  double F[4];  // the wave's class of P_inv
#pragma unroll
  for (int k = 0; k < 4; k++) F[k] = a.pc[(c.w * 4 + k) * 64 + c.lane];
  for (int i = tid; i < TAB; i += WGS) s.tab[i] = i < a.n_codes ? a.A.etab[i] : 0.0;
  if (tid == 0) s.bad = 0;
  auto tot = [&](int k) __attribute__((always_inline)) { return uni(s.tot[k]); };
  for (;;) {
    if (tid == 0)
      s.ticket = __hip_atomic_fetch_add(a.ctl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int tk = uni(s.ticket);
    if (tk >= a.n_tickets || c.dead) break;
    int id = 0;
    if (a.task) {
      int hi = a.n_tasks;  // the last task whose first ticket is not beyond this one
      while (hi - id > 1) {
        const int mid = (id + hi) >> 1;
        if (uni(a.task[mid].ticket0) <= tk) id = mid;
        else hi = mid;
      }
      const int *f = reinterpret_cast<const int *>(a.task + id);
      int *to = reinterpret_cast<int *>(&c.t);
#pragma unroll
      for (int i = 0; i < (int)(sizeof(TeamTask) / sizeof(int)); i++) to[i] = uni(f[i]);
    } else {
      c.t = a.one;
    }
    const TeamTask &t = c.t;
    c.rank = tk - t.ticket0;
    c.b0 = t.b0 + c.rank * t.bpw;
    c.nb = min(t.bpw, t.nb - c.rank * t.bpw);
    c.slots = a.slots + (size_t)t.slot0 * TEAM_SLOT_WORDS;
    c.halo0 = a.halo + (long)HALO_BLOCK * t.b0;
    c.copies = team_copies(t.nwg);
    c.copy = c.rank % c.copies;
    c.slab = 2 * TEAM_NQ * t.nwg;
    c.ep = c.zp = 0;
    c.lay_out();

    const bool mr = KIND == MEAN_ROW && t.mean_row >= 0;
    // the state's constants, and the state itself (every thread keeps and
    // advances it from the same totals)
    const Scal *st = a.st + id;
    const bool l2 = KIND == PLAIN || (KIND == MEAN_ROW && uni(st->norm));
    const int max_iter = uni(st->max_iter), max_restarts = uni(st->max_restarts);
    const bool confirm = uni(st->rep_factor) > 0.0;
    const double eps = uni(st->eps), tol_abs = uni(st->tol_abs), tol_rel = uni(st->tol_rel), bd_tol = uni(st->bd_tol);
    double err = 0.0, err0 = 0.0, size_opt = 0.0, err_rep = 0.0, rho = 0.0, target = 0.0;
    int iter = 0, restarts = 0, n_rep = 0;
    bool done = false, converged = false, improved = false;

    double r[T][4], rhat[T][4], p[T][4], nu[T][4], x[T][4];
    double hh = 0.0, alpha = 0.0, omega = 1.0, mean = 0.0;
    const bool prof = a.phase && c.rank == 0 && wave_id() == 0;
    auto lap = [&](int k) __attribute__((always_inline)) {
      if (__builtin_expect(prof, 0) && tid == 0) {
        const u64 now = wall_clock64();
        s.phase[k] += now - s.tick;
        s.tick = now;
      }
    };
    if (prof && tid == 0) {
      for (int k = 0; k < TEAM_PHASES; k++) s.phase[k] = 0;
      s.tick = wall_clock64();
    }
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
#pragma unroll
      for (int k = 0; k < 4; k++)  // the caller's arrays: 8-byte aligned; x0's NaNs are made quiet (EMPTY is none)
        x[tt][k] = __builtin_canonicalize(a.x0[c.cell(tt) + k]);
      if (c.ok(tt)) st4(a.xopt, c.cell(tt), x[tt]);
      else x[tt][0] = x[tt][1] = x[tt][2] = x[tt][3] = 0.0;
    }
    CELLS r[tt][k] = rhat[tt][k] = p[tt][k] = nu[tt][k] = 0.0;
    {  // the whole team is here and its words of z are empty before any is awaited
      c.clear();
      c.clear();
      double v[2] = {0.0, 0.0};
      c.template exchange<2, false>(v, -a.form_polls);
    }

    // y = A z; the mean row: sum h^2 z in v[2], the other factor's value there in v[3]
    double z[T][4], y[T][4];
    auto mean_row = [&](double (&v)[4], const double (&other)[T][4]) __attribute__((always_inline)) {
      if constexpr (KIND == MEAN_ROW)
        if (mr) CELLS {
          v[2] += s.h2[c.lb(tt)] * z[tt][k];
          if (c.ok(tt) && c.cell(tt) + k == t.mean_row) {
            y[tt][k] = 0.0;
            v[3] = other[tt][k];
          }
        }
    };
    auto put_mean_row = [&]() __attribute__((always_inline)) {
      if (mr) CELLS if (c.ok(tt) && c.cell(tt) + k == t.mean_row) y[tt][k] = tot(2);
    };
    auto keep = [&]() __attribute__((always_inline)) {  // the iterate is the best so far
#pragma unroll
      for (int tt = 0; tt < T; tt++)
        if (c.ok(tt)) st4(a.xopt, c.cell(tt), x[tt]);
    };
    auto recall = [&]() __attribute__((always_inline)) {  // go on with the best one
#pragma unroll
      for (int tt = 0; tt < T; tt++)
        if (c.ok(tt)) ld4(a.xopt, c.cell(tt), x[tt]);
    };
    // the size of the residual as it is compared: |r|^2 or |r|_inf
    auto norm_of = [l2](double v) { return l2 ? sqrt(v) : v; };
    double beta = 0.0;
    bool restart = false, replace = false;
    // The state at the top of an iteration (kernels.h evaluate: the same
    // rules, without the projection and the stall window); rho and beta are
    // the new ones.
    auto assess = [&](double rr, double size) __attribute__((always_inline)) {
      iter++;
      improved = size < size_opt;
      restart = replace = false;
      if (improved) size_opt = size;
      if (__builtin_expect(improved && size <= target, 0)) {
        err = uni(norm_of(size));
        if (err <= tol_abs || err / err0 <= tol_rel) {
          if (confirm) replace = true;  // the recurrence says converged: confirm it on the residual itself
          else converged = done = true;
        }
      }
      // (a claim made in the last iteration is still confirmed)
      if (iter >= max_iter && !replace) (a.start == TEAM_REFINES ? replace : done) = true;
      const bool breakdown = rho * rho < bd_tol * rr * hh || !(fabs(beta) < 1e30);
      if (__builtin_expect(breakdown && !done && !replace && max_restarts > 0, 0)) {
        restarts++;
        if (restarts >= max_restarts) {
          (a.start == TEAM_REFINES ? replace : done) = true;
        } else {
          restart = true;
          hh = rho = rr;  // rhat = r
        }
      }
    };

    // Residuals r = b - A x (the start, and the confirmations of a mixed
    // solve), each followed by iterations.
    for (;;) {
      c.place();
      CELLS z[tt][k] = x[tt][k];
      c.spmv(z, y, TEAM_POLLS);
      lap(0);
      if constexpr (KIND == MEAN_ROW) {
        double v[4] = {};
        mean_row(v, z);
        c.template exchange<4, false>(v, TEAM_POLLS);
        if (c.dead) break;
        put_mean_row();
      }
      {
        double f[KIND == PLAIN ? 1 : 2] = {};
#pragma unroll
        for (int tt = 0; tt < T; tt++) {
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const double bb = a.b[c.cell(tt) + k];
            const bool row0 = mr && c.cell(tt) + k == t.mean_row;  // b = 0 there (ExpAMRSolver.cpp:340-345)
            const double ri = c.ok(tt) ? (row0 ? 0.0 : bb) - y[tt][k] : 0.0;
            r[tt][k] = rhat[tt][k] = p[tt][k] = ri;
            f[0] += ri * ri;
            if constexpr (KIND != PLAIN) f[1] = nmax(f[1], fabs(ri));
          }
        }
        c.place();
        c.template exchange<KIND == PLAIN ? 1 : 2, KIND != PLAIN>(f, TEAM_POLLS);
      }
      if (c.dead) break;
      c.clear();
      const double size = l2 ? tot(0) : tot(1);
      err = uni(norm_of(size));
      if (replace) {
        n_rep++;
        if (a.start == TEAM_REFINES) {  // the next pass counts its own
          if (tid == 0) s.restarts += restarts;
          restarts = 0;
        }
      } else {
        err0 = err;
        // sizes above this have not converged (the test itself is exact)
        const double most = fmax(tol_abs, tol_rel * err0) * (1.0 + 1e-9);
        target = uni(l2 ? most * most : most);
      }
      size_opt = size;
      err_rep = err;
      hh = rho = tot(0);
      improved = replace;
      done = err == 0.0 || iter >= max_iter;
      if (replace && (err <= tol_abs || err / err0 <= tol_rel)) converged = done = true;
      if (a.start != TEAM_PLAIN) {
        if (err != err || err > 1.79e308) {
          done = true;
          converged = false;
        } else if (!replace && (err == 0.0 || (a.start >= TEAM_ACCEPTS && (err <= tol_abs || tol_rel >= 1.0)))) {
          converged = done = true;
        }
      }
      if (n_rep >= TEAM_MAX_CONFIRM) done = true;
      if (!done && improved) keep();
      if (done && !improved) recall();
      lap(4);
      if (done) break;
      beta = 0.0;
      bool pending = false;  // the last iteration's r is yet to be assessed
      for (;;) {
        // nu = A P p and alpha.  The size of r, by which the iteration before
        // is assessed, is summed with (rhat, nu), one exchange an iteration
        // less; the mean row's own sums take its place there.
        c.place();
        CELLS z[tt][k] = p[tt][k];
        c.prec(F, z);
        lap(1);
        c.place();
        c.spmv(z, y, TEAM_POLLS);
        double coef, by_row = 0.0;
        {
          double v[KIND == PLAIN ? 2 : KIND == NORM_MAX ? 3 : 4] = {};
          if constexpr (KIND == MEAN_ROW) mean_row(v, rhat);
          CELLS {
            v[0] += y[tt][k] * rhat[tt][k];
            if constexpr (KIND != MEAN_ROW) v[1] += r[tt][k] * r[tt][k];
            if constexpr (KIND == NORM_MAX) v[2] = nmax(v[2], fabs(r[tt][k]));
          }
          lap(0);
          c.place();
          c.template exchange<KIND == PLAIN ? 2 : KIND == NORM_MAX ? 3 : 4, KIND == NORM_MAX>(v, TEAM_POLLS);
        }
        if (c.dead) break;
        lap(3);
        if constexpr (KIND == MEAN_ROW) {
          if (mr) by_row = tot(3) * tot(2);
          put_mean_row();
        } else if (pending) {
          assess(tot(1), tot(l2 ? 1 : 2));
          if (__builtin_expect(done || replace || restart, 0)) {  // nothing of this pass is kept
            c.clear();
            if (!restart) {
              if (!improved) recall();
              break;
            }
            if (improved) keep();
            CELLS rhat[tt][k] = p[tt][k] = r[tt][k];
            pending = false;
            continue;
          }
          if (improved) keep();
        }
        alpha = coef = uni(rho / (tot(0) + by_row + eps));
        CELLS {  // s = r - alpha nu; x follows
          x[tt][k] = x[tt][k] + coef * z[tt][k];
          r[tt][k] = r[tt][k] - coef * y[tt][k];
          nu[tt][k] = y[tt][k];
        }
        c.clear();
        lap(2);
        // t = A P s and omega
        c.place();
        CELLS z[tt][k] = r[tt][k];
        c.prec(F, z);
        lap(1);
        c.place();
        c.spmv(z, y, TEAM_POLLS);
        {
          double v[4] = {};
          if constexpr (KIND == MEAN_ROW) mean_row(v, r);
          CELLS {
            v[0] += y[tt][k] * r[tt][k];
            v[1] += y[tt][k] * y[tt][k];
            if constexpr (KIND != MEAN_ROW) {
              v[2] += y[tt][k] * rhat[tt][k];
              v[3] += r[tt][k] * rhat[tt][k];
            }
          }
          lap(0);
          c.place();
          c.template exchange<4, false>(v, TEAM_POLLS);
        }
        if (c.dead) break;
        lap(3);
        double ts = tot(0), tq = tot(1);
        if constexpr (KIND == MEAN_ROW) {
          if (mr) {
            ts += tot(2) * tot(3);
            tq += tot(2) * tot(2);
          }
          put_mean_row();
        }
        omega = coef = uni(ts / (tq + eps));
        CELLS {  // r = s - omega t
          x[tt][k] = x[tt][k] + coef * z[tt][k];
          r[tt][k] = r[tt][k] - coef * y[tt][k];
        }
        const double aow = alpha / (omega + eps);
        if constexpr (KIND == MEAN_ROW) {
          double f[3] = {};
          CELLS {
            const double rd = r[tt][k];
            f[0] += rd * rd;
            f[1] += rhat[tt][k] * rd;
            f[2] = nmax(f[2], fabs(rd));
          }
          lap(2);
          c.place();
          c.template exchange<3, true>(f, TEAM_POLLS);
          if (c.dead) break;
          lap(3);
          beta = uni((tot(1) / (rho + eps)) * aow);
          rho = tot(1);
          assess(tot(0), tot(l2 ? 0 : 2));
          c.clear();
          if (improved && !done && !replace) keep();
          if (!improved && (done || replace)) recall();
          if (done || replace) break;
          if (restart) {
            CELLS rhat[tt][k] = p[tt][k] = r[tt][k];
            continue;
          }
        } else {
          // rhat r of r = s - omega t, from this exchange's sums
          const double rhr = tot(3) - omega * tot(2);
          beta = uni((rhr / (rho + eps)) * aow);
          rho = uni(rhr);
          pending = true;
          c.clear();
        }
        CELLS p[tt][k] = r[tt][k] + beta * (p[tt][k] - omega * nu[tt][k]);
        lap(2);
      }
      if (c.dead || done) break;
    }
    if (!c.dead) {  // the h^2-weighted mean removed (ExpAMRSolver.cpp:383-415)
      double v[2] = {};
      CELLS {
        const double w2 = s.h2[c.lb(tt)];
        v[0] += x[tt][k] * w2;
        v[1] += w2;
      }
      c.place();
      c.template exchange<2, false>(v, TEAM_POLLS);
      mean = tot(0) / tot(1);
#pragma unroll
      for (int tt = 0; tt < T; tt++)
        if (c.ok(tt) && !c.dead)
#pragma unroll
          for (int k = 0; k < 4; k++) a.out[c.cell(tt) + k] = x[tt][k] - mean;
    }
    if (c.dead) break;
    lap(4);
    if (c.rank == 0 && tid == 0) {
      Scal *o = a.st + id;
      o->iter = iter;
      o->restarts = s.restarts + restarts;
      o->n_rep = n_rep;
      o->converged = converged;
      o->improved = improved;
      o->done = o->idle = 1;
      o->err0 = err0;
      o->err = o->err_opt = l2 ? sqrt(size_opt) : size_opt;
      o->err_rep = err_rep;
      o->mean = mean;
      __hip_atomic_fetch_add(a.ctl + 2, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (prof)
        for (int k = 0; k < TEAM_PHASES; k++) a.phase[(size_t)id * TEAM_PHASES + k] = s.phase[k];
    }
    __syncthreads();  // the shared state is rewritten by the next task
  }
}

template <int KIND>
const void *shape_kernel(int shape) {
  return shape == TEAM_16   ? reinterpret_cast<const void *>(&k_team<256, 1, KIND>)
         : shape == TEAM_32 ? reinterpret_cast<const void *>(&k_team<512, 1, KIND>)
         : shape == TEAM_48 ? reinterpret_cast<const void *>(&k_team<768, 1, KIND>)
                            : reinterpret_cast<const void *>(&k_team<512, 2, KIND>);
}
const void *shape_kernel(int shape, int kind) {
  return kind == PLAIN ? shape_kernel<PLAIN>(shape) : kind == NORM_MAX ? shape_kernel<NORM_MAX>(shape) : shape_kernel<MEAN_ROW>(shape);
}
int shape_threads(int shape) { return shape == TEAM_64 ? 512 : 16 * team_blocks(shape); }
size_t shape_lds(int shape) {
  return shape == TEAM_16 ? sizeof(Shared<256, 1>) : shape == TEAM_32 ? sizeof(Shared<512, 1>) : shape == TEAM_48 ? sizeof(Shared<768, 1>) : sizeof(Shared<512, 2>);
}

}  // namespace

int team_resident(int shape) {
  static std::atomic<int> known[64][TEAM_SHAPES];  // per device: looked up once (0: not yet)
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (const int n = known[dev][shape].load()) return n;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  int least = 1 << 30;
  for (int kind = 0; kind < KINDS; kind++) {
    const void *k = shape_kernel(shape, kind);
    int per = 0;
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shape_lds(shape)) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, shape_threads(shape), shape_lds(shape)) != hipSuccess)
      return 0;
    least = per < least ? per : least;
  }
  known[dev][shape] = cus * least;
  return cus * least;
}

hipError_t team_launch(const TeamArgs &a, int shape, size_t n_words, int grid, hipStream_t stream) {
  TeamArgs args = a;
  hipError_t e = hipMemsetAsync(a.slots, 0, n_words * sizeof(u64), stream);
  if (e == hipSuccess) e = hipMemsetAsync(a.ctl, 0, 3 * sizeof(int), stream);
  if (e != hipSuccess) return e;
  void *params[] = {&args};
  return hipLaunchCooperativeKernel(shape_kernel(shape, a.mean_rows ? MEAN_ROW : a.norm_max ? NORM_MAX : PLAIN), dim3(grid), dim3(shape_threads(shape)),
                                    params, (unsigned)shape_lds(shape), stream);
}

}  // namespace cup2d
