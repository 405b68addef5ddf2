// hes_resident.hpp -- the time loop of one problem in one launch, its state on
// the chip from the first step to the last.
//
// A step needs the maximum CFL speed of the whole state, so a launch per step
// (k_step) streams every state through memory and pays a launch and its ramp
// per step: 5.5 us per step at 1000 cells (Rusanov), 20.1 us at 2^18, of which
// the arithmetic is 2 and 4.  Here a team of workgroups, all resident at once,
// holds the problem: one cell per lane in registers for the whole run.
//
//   wave       64 consecutive cells; lanes 1..62 are updated by this wave,
//              lanes 0 and 63 copy the neighbour waves' cells through LDS
//   workgroup  `own` cells and `halo` cells on either side that a neighbour
//              workgroup owns; the copies are stepped along with the own
//              cells (the same arithmetic on the same values), lose one
//              valid cell per step at their outer end, and are renewed from
//              the neighbour every `halo` steps
//   team       per step each workgroup publishes the maximum of its own
//              cells' speeds in a slot of its own and reads all the others
//
// Two messages cross workgroups, both as single 64-bit words that carry their
// own arrival mark, so no fence and no second round trip is needed: the
// maximum's sign bit alternates with the use of its slot, and a halo word is
// 32 bits of a value beside a 32-bit tag.  A slot (two by step parity) is
// written again only after every workgroup has published the step between,
// i.e. has read it.
//
// Every wait gives up after ResTeam::wait, or at once when another workgroup
// has: the launch then ends without a result and the caller's input is whole
// (results go to another buffer, and only after the last wait).
//
// Measured (two phases: see plan_resident), single phase, 65 pieces, us per
// step, one launch per step (replayed from a graph) against this: 1000 cells
// 5.5 -> 3.6 (Rusanov) and 6.2 -> 3.8 (HLL), 30011 cells 7.7 -> 4.0 and 8.5 ->
// 3.8, 2^18 cells 20.1 -> 9.4 and 21.6 -> 11.8.  What is left: the chain of
// dependent FP64 operations of one cell (2.2 us Rusanov, 2.9 HLL: one workgroup,
// which exchanges nothing), the team's exchange (1.1 us more with 2 workgroups,
// 1.4 with 5, 2.2 with 256; with HLL, whose mid state falls into the wait, 0.8 to
// 0.9), and from two waves per SIMD on the FP64 issue rate (0.95 us per tile and
// SIMD).
#pragma once
#include <algorithm>
#include <type_traits>
#include <vector>
#include "hes_step.hpp"

namespace hes {

constexpr int RES_SLOT = 8;  // 64-bit words per slot: one per 64 B (stores of many
                             // workgroups into one line serialise; 256 workgroups: 3.1 -> 2.1 us)
constexpr long long RES_WAIT_US = 4000000;  // the longest wait for a message, unless the user sets it
constexpr int RES_POLLS = 64;               // polls between two looks at the time
constexpr int RES_HALO = 8;  // halo cells on either side of a workgroup (a team of one has none)

// wave_max by DPP shifts instead of the LDS crossbar (a dependent chain of 6
// moves and maxima, no ds_bpermute round trips): the maximum in every lane.
template <int CTRL>
__device__ __forceinline__ double dpp_max(double v) {
  return fmax(v, dpp_shift<CTRL>(v));
}
__device__ __forceinline__ double wave_max_dpp(double v) {
  v = dpp_max<0x111>(v);  // row_shr:1, 2, 4, 8: the rows of 16 lanes
  v = dpp_max<0x112>(v);
  v = dpp_max<0x114>(v);
  v = dpp_max<0x118>(v);
  v = dpp_max<0x142>(v);  // row_bcast:15, 31: across the rows, into lane 63
  v = dpp_max<0x143>(v);
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// One workgroup's share of a problem, and the team's message buffers.
struct ResTeam {
  const double* __restrict__ Qin;
  double* __restrict__ Qout;
  double* __restrict__ Cout;
  long long pitch, lo, hi;  // the problem's cells
  int G, rank, own;         // workgroups, this one, its cells (at least RES_HALO for G > 1)
  double cfl, dx, t, t_end;
  long long kmax;           // steps at most
  double* dt_hist;          // optional: dt of every step
  int* status;
  int lxf;
  unsigned long long* slots;   // 2 G RES_SLOT words, zero at the start
  unsigned long long* border;  // halo words: 2 G 2 RES_HALO 2 NC
  unsigned tag0;               // larger than every tag in `border`
  int* gave_up;                // nonzero: a wait ended without its message
  long long wait;              // ticks of the 100 MHz counter; 0: the team's last workgroup
                               // gives up in place of its first wait
};

struct ResOut {
  long long steps;
  double t, lmax;
  bool ok;
};

__device__ __forceinline__ void res_store(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long res_load(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Barrier of the workgroup for LDS traffic alone: __syncthreads would also wait
// for the messages on their way to memory.
__device__ __forceinline__ void res_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// One check of a wait's end, every few polls: true when the wait is over
// without its message (the time is up here, or another workgroup gave up).
__device__ __forceinline__ bool res_expired(const ResTeam& a, int& polls, long long& since) {
  if (++polls % RES_POLLS) return false;
  const long long now = wall_clock64();
  if (since == 0) since = now;
  if (__hip_atomic_load(a.gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return true;
  if (now - since < a.wait) return false;
  __hip_atomic_store(a.gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// Whether this workgroup gives up before it waits at all: with no time to wait
// the team's last one does.  Asked once, before the steps: a test of the time in
// every exchange took up to 0.07 us per step at 1000 cells.
__device__ __forceinline__ bool res_quits(const ResTeam& a) {
  const bool quits = a.wait == 0 && a.G > 1 && a.rank == a.G - 1;
  if (quits && threadIdx.x == 0)
    __hip_atomic_store(a.gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return quits;
}

// The team's maximum of step s: publish this workgroup's, then wait for all
// (one wave, every lane active).  A state without a positive speed (NaN) still
// publishes a non-zero word.
__device__ __forceinline__ void res_publish(const ResTeam& a, long long s, double m) {
  const unsigned long long sign = (unsigned long long)((s >> 1) & 1) << 63;
  const unsigned long long bits = m > 0.0 ? (unsigned long long)__double_as_longlong(m) : 1ull;
  if ((threadIdx.x & 63) == 0)
    res_store(a.slots + ((s & 1) * a.G + a.rank) * (long long)RES_SLOT, bits | sign);
}
// LEAD: leader receives the first workgroup that attains it.
template <int MAXG, bool LEAD = false>
__device__ __forceinline__ bool res_collect(const ResTeam& a, long long s, double& lmax,
                                            int* leader = nullptr) {
  const int lane = threadIdx.x & 63;
  const unsigned long long sign = (unsigned long long)((s >> 1) & 1) << 63;
  const unsigned long long* sl = a.slots + (s & 1) * a.G * (long long)RES_SLOT;
  int polls = 0;
  long long since = 0;
  for (;;) {
    unsigned long long x[MAXG / 64];
#pragma unroll
    for (int k = 0; k < MAXG / 64; ++k) {
      x[k] = sign | 1ull;
      if (64 * k < a.G) {  // uniform; the loads of all slots are in flight together
        const int b = 64 * k + lane;
        x[k] = res_load(sl + (long long)(b < a.G ? b : a.rank) * RES_SLOT);
      }
    }
    bool here = true;
    double m = 0.0;
#pragma unroll
    for (int k = 0; k < MAXG / 64; ++k) {
      here = here && x[k] != 0ull && ((x[k] ^ sign) >> 63) == 0ull;
      m = fmax(m, __longlong_as_double((long long)(x[k] & 0x7fffffffffffffffull)));
    }
    if (__all(here)) {
      lmax = wave_max_dpp(m);
      if constexpr (LEAD) {
        *leader = 0;
#pragma unroll
        for (int k = MAXG / 64 - 1; k >= 0; --k) {
          const unsigned long long at = __ballot(
              64 * k + lane < a.G &&
              __longlong_as_double((long long)(x[k] & 0x7fffffffffffffffull)) == lmax);
          if (at) *leader = 64 * k + (int)__builtin_ctzll(at);
        }
      }
      return true;
    }
    if (res_expired(a, polls, since)) return false;
  }
}

typedef unsigned __attribute__((may_alias)) u32_any;

// Halo words of the cells a workgroup shares with its neighbours, renewed at
// every RES_HALO-th step from and into LDS (word k of a side: 32-bit half k of
// its RES_HALO cells' states): side 0 is read by the left neighbour (this
// workgroup's first cells), side 1 by the right one (its last cells).  One
// wave each, every lane active.
template <int NC>
__device__ __forceinline__ unsigned long long* res_words(const ResTeam& a, long long round,
                                                         int rank, int side) {
  return a.border + (((round & 1) * a.G + rank) * 2 + side) * (long long)(RES_HALO * 2 * NC);
}
template <int NC>
__device__ __forceinline__ void res_send(const ResTeam& a, long long round, unsigned tag, int side,
                                         const double* cells) {
  unsigned long long* w = res_words<NC>(a, round, a.rank, side);
  const u32_any* src = (const u32_any*)cells;
#pragma unroll 1
  for (int k = threadIdx.x & 63; k < RES_HALO * 2 * NC; k += 64)
    res_store(w + k, (unsigned long long)src[k] | ((unsigned long long)tag << 32));
}
template <int NC>
__device__ __forceinline__ bool res_receive(const ResTeam& a, long long round, unsigned tag,
                                            int rank, int side, double* cells) {
  const unsigned long long* w = res_words<NC>(a, round, rank, side);
  u32_any* dst = (u32_any*)cells;
  constexpr int N = RES_HALO * 2 * NC, M = (N + 63) / 64;
  const int lane = threadIdx.x & 63;
  int polls = 0;
  long long since = 0;
  for (;;) {
    unsigned long long x[M];
#pragma unroll
    for (int k = 0; k < M; ++k) x[k] = res_load(w + (64 * k + lane < N ? 64 * k + lane : lane));
    bool here = true;
#pragma unroll
    for (int k = 0; k < M; ++k) here = here && (unsigned)(x[k] >> 32) == tag;
    if (__all(here)) {
#pragma unroll
      for (int k = 0; k < M; ++k)
        if (64 * k + lane < N) dst[64 * k + lane] = (unsigned)x[k];
      return true;
    }
    if (res_expired(a, polls, since)) return false;
  }
}

// The run of one workgroup, single phase.  T: tiles of 64 lanes that a wave
// holds (its registers); MAXG: the largest team it is built for (a multiple
// of 64).  Per step the thermodynamic state of a cell is formed once, for its
// flux and for its speed (k_step forms it twice, for the state it reads and
// the one it writes); with one tile per wave and registers to keep it, the
// flux, and always HLL's mid state, fall into the wait for the team's maximum.
// hook: told of every state s that the run passes through, once its maximum
// lmax is known: hook.tile for each of a wave's tiles (every lane active; own:
// the lane's cell i belongs to this workgroup; lead: this is the team's first
// workgroup with a cell of speed lmax), then hook.end.
struct ResNoHook {};
template <int FLUX, int FAST, int BLK, int T, int MAXG, bool FLUX_LDS = false, class Hook = ResNoHook>
__device__ __forceinline__ ResOut resident_run1(const ResTeam& a, const MatDev& mat,
                                                Hook hook = Hook()) {
  constexpr int NC = 14, W = BLK / 64, NT = W * T;
  constexpr bool HOOK = !std::is_same<Hook, ResNoHook>::value;
  constexpr bool LATE_FLUX = T == 1;
  __shared__ double edge[2][NT][2][NC];  // new first and last updated cell of every tile, by parity
  __shared__ double red[2][W];           // every wave's maximum, by parity
  __shared__ double mine_out[2][RES_HALO][NC], theirs[2][RES_HALO][NC];
  // FLUX_LDS: the 11 components of every cell's flux that are not zero
  __shared__ double flux[FLUX_LDS ? NT : 1][FLUX_LDS ? 11 : 1][64];
  __shared__ double team_max, tnow[2];
  __shared__ int dead, leader;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long o0 = a.lo + (long long)a.rank * a.own;
  const long long o1 = o0 + a.own < a.hi ? o0 + a.own : a.hi;
  // positions are counted from the workgroup's first own cell
  const int n_own = (int)(o1 - o0);
  const int n_lo = o0 - a.lo < (1 << 24) ? (int)(a.lo - o0) : -(1 << 24);  // the problem's first cell
  const int n_hi = a.hi - o0 < (1 << 24) ? (int)(a.hi - o0) : 1 << 24;     // and past its last
  const int halo = a.G > 1 ? RES_HALO : 0;
  auto cell = [&](int k) { return TILE * (w * T + k) + lane - halo; };
  auto mine = [&](int k) {
    const int tile = w * T + k, j = cell(k);
    return (lane >= 1 || (tile == 0 && halo == 0)) && (lane <= TILE || (tile == NT - 1 && halo == 0)) &&
           j >= 0 && j < n_own;
  };
  double q[T][NC], c[T];
#pragma unroll
  for (int k = 0; k < T; ++k) {
    const int j = cell(k), jc = j < n_lo ? n_lo : (j >= n_hi ? n_hi - 1 : j);
#pragma unroll
    for (int r = 0; r < NC; ++r) q[k][r] = a.Qin[r * a.pitch + o0 + jc];
  }
  if (threadIdx.x == 0) {
    dead = 0;
    leader = 0;
  }
  const bool quits = res_quits(a);
  double t = a.t, lmax = 0.0;
  long long s = 0;
  int to_halo = RES_HALO;
  int bad = 0;
  bool ok = true;
  for (;; ++s) {
    double f[T][NC], u1[T], mn[T], mx[T], m = 0.0;
    Thermo th;
#pragma unroll
    for (int k = 0; k < T; ++k) {
      thermo<true, FAST>(mat, 1.0, q[k], th);
      c[k] = sound_speed(mat, th);
      u1[k] = th.u[0];
      const bool own = mine(k);
      bad |= own && (th.bad | !(c[k] < 1e300));
      m = fmax(m, own ? fabs(u1[k]) + c[k] : 0.0);
      if (!LATE_FLUX) phase_flux(mat, 1.0, th, q[k] + 5, f[k]);
      if (FLUX_LDS) {
#pragma unroll
        for (int r = 0, z = 0; r < NC; ++r)
          if (r < 5 || (r - 5) % 3) flux[w * T + k][z++][lane] = f[k][r];
      }
    }
    m = wave_max_dpp(m);
    if (lane == 0) red[s & 1][w] = m;
    res_barrier();
    lmax = wave_max_dpp(lane < W ? red[s & 1][lane] : 0.0);
    if (a.G > 1 && w == 0) res_publish(a, s, lmax);
    if (LATE_FLUX) phase_flux(mat, 1.0, th, q[0] + 5, f[0]);
    if (FLUX == FLUX_HLL) {
#pragma unroll
      for (int k = 0; k < T; ++k) mid_range1<FAST>(mat, q[k], mn[k], mx[k]);
    }
    if (a.G > 1) {
      if (w == 0) {
        double lm = 0.0;
        int lead = 0;
        const bool got = !quits && res_collect<MAXG, HOOK>(a, s, lm, &lead);
        if (lane == 0) {
          team_max = lm;
          if (HOOK) leader = lead;
          if (!got) dead = 1;
        }
      }
      res_barrier();
      lmax = team_max;
      if (dead) {
        ok = false;
        break;
      }
    }
    if constexpr (HOOK) {
#pragma unroll
      for (int k = 0; k < T; ++k)
        hook.tile(s, lmax, mine(k), leader == a.rank, o0 + cell(k), q[k], c[k], u1[k]);
      hook.end(s, lmax);
    }
    if (s >= a.kmax || !(t < a.t_end)) break;  // main.jl:202 `while t < T`
    const double dtdx = a.cfl * rcp(lmax);
    if (w == 0) {  // the time, by one wave
      const double dt = a.cfl * a.dx / lmax;  // main.jl:212
      if (lane == 0) {
        if (a.dt_hist && a.rank == 0) a.dt_hist[s] = dt;
        tnow[s & 1] = t + dt;
      }
    }
    const bool renew = a.G > 1 && --to_halo == 0;  // uniform
#pragma unroll
    for (int k = 0; k < T; ++k) {
      const double smin = u1[k] - c[k], smax = u1[k] + c[k];
      if (FLUX_LDS) {
#pragma unroll
        for (int r = 0, z = 0; r < NC; ++r) f[k][r] = r < 5 || (r - 5) % 3 ? flux[w * T + k][z++][lane] : 0.0;
      }
      double upd[NC];
      if (FLUX == FLUX_RUSANOV)
        update_rusanov1<true>(q[k], f[k], smin, smax, dtdx, a.lxf, upd);
      else
        update_hll1<true>(q[k], f[k], hll_coef(mn[k], mx[k], smin, lane_down(smax)), dtdx, upd);
      // cells beyond the right halo stay as they are: copies that nothing renews
      const int j = cell(k);
      if (lane >= 1 && lane <= TILE && j > n_lo && j < n_hi - 1 && j < n_own + halo) {
#pragma unroll
        for (int r = 0; r < NC; ++r) q[k][r] = upd[r];
      }
      if (lane == 1 || lane == TILE) {
        double* e = edge[s & 1][w * T + k][lane == 1 ? 0 : 1];
#pragma unroll
        for (int r = 0; r < NC; ++r) e[r] = q[k][r];
      }
      if (renew && mine(k)) {
        if (j < RES_HALO) {
#pragma unroll
          for (int r = 0; r < NC; ++r) mine_out[0][j][r] = q[k][r];
        }
        if (j >= n_own - RES_HALO) {
#pragma unroll
          for (int r = 0; r < NC; ++r) mine_out[1][j - (n_own - RES_HALO)][r] = q[k][r];
        }
      }
    }
    res_barrier();
    t = tnow[s & 1];
#pragma unroll
    for (int k = 0; k < T; ++k) {
      const int tile = w * T + k;
      if ((lane == 0 && tile > 0) || (lane == 63 && tile < NT - 1)) {
        const double* e = edge[s & 1][lane == 0 ? tile - 1 : tile + 1][lane == 0 ? 1 : 0];
#pragma unroll
        for (int r = 0; r < NC; ++r) q[k][r] = e[r];
      }
    }
    if (renew) {
      to_halo = RES_HALO;
      const long long round = (s + 1) / RES_HALO;
      const unsigned tag = a.tag0 + (unsigned)s;
      bool got = true;
      if (w == 0 && a.rank > 0) {
        res_send<NC>(a, round, tag, 0, &mine_out[0][0][0]);
        got = res_receive<NC>(a, round, tag, a.rank - 1, 1, &theirs[0][0][0]);
      }
      if (w == W - 1 && a.rank < a.G - 1) {
        res_send<NC>(a, round, tag, 1, &mine_out[1][0][0]);
        got = res_receive<NC>(a, round, tag, a.rank + 1, 0, &theirs[1][0][0]);
      }
      if (!got) dead = 1;  // seen after the next step's barriers
      res_barrier();
#pragma unroll
      for (int k = 0; k < T; ++k) {
        const int j = cell(k);
        const bool left = j < 0 && j >= n_lo;
        if (left || (j >= n_own && j < n_own + RES_HALO && j < n_hi)) {
          const double* e = left ? theirs[0][j + RES_HALO] : theirs[1][j - n_own];
#pragma unroll
          for (int r = 0; r < NC; ++r) q[k][r] = e[r];
        }
      }
    }
  }
  if (ok) {
#pragma unroll
    for (int k = 0; k < T; ++k) {
      if (mine(k)) {
        const long long i = o0 + cell(k);
#pragma unroll
        for (int r = 0; r < NC; ++r) a.Qout[r * a.pitch + i] = q[k][r];
        a.Cout[i] = c[k];
      }
    }
    if (__any(bad) && lane == 0) atomicOr(a.status, 1);
  }
  return {s, t, lmax, ok};
}

// The run of one workgroup, two phases: four waves, one per SIMD, of TW cells
// each (lanes TW and up repeat the last one in the stages of one lane per
// cell).  The state's home is LDS, since the faces with a volume-fraction jump
// are worked on by groups of GL lanes (face_path2, face_path2_hll) that need
// the states of any face of the wave, and since their quadrature leaves no
// registers for it.  A diffused interface soon makes every face of a small
// problem such a face, and a face's 6 (Rusanov) or 18 (HLL) nodes are the
// longest chain of a step: with TW = 16 all faces of a wave run at once, and a
// problem of 1000 cells spreads over 24 workgroups; larger problems take wider
// tiles (more of a problem on the chip, more faces per wave in turn).  GL is
// that of the step-by-step kernels, whose sums over the nodes it orders.  All
// face terms but Lax-Friedrichs' fall into the wait for the team's maximum.
template <int FLUX, int FAST, int TW, int MAXG>
__device__ __forceinline__ ResOut resident_run2(const ResTeam& a, const MatDev* mat, double relax,
                                                double relax_p) {
  constexpr int NC = 30, W = 4, STEP = TW - 2;
  constexpr int GL = FLUX == FLUX_HLL ? HES_PATH_HLL_LANES : HES_PATH_LANES;
  __shared__ double cells[W][NC][TW];   // the state
  __shared__ double path[W][NC][TW];    // jump faces: flux difference (HLL), then the path terms
  __shared__ double bound[W][3][TW];    // HLL: s_l, s_r, 1 / (s_r - s_l) of the faces
  __shared__ unsigned char list[W][64]; // the wave's jump faces
  __shared__ double red[2][W];
  __shared__ double mine_out[2][RES_HALO][NC], theirs[2][RES_HALO][NC];
  __shared__ double team_max, tnow[2];
  __shared__ int dead;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane < TW ? lane : TW - 1;
  const long long o0 = a.lo + (long long)a.rank * a.own;
  const long long o1 = o0 + a.own < a.hi ? o0 + a.own : a.hi;
  // positions are counted from the workgroup's first own cell
  const int n_own = (int)(o1 - o0);
  const int n_lo = o0 - a.lo < (1 << 24) ? (int)(a.lo - o0) : -(1 << 24);
  const int n_hi = a.hi - o0 < (1 << 24) ? (int)(a.hi - o0) : 1 << 24;
  const int halo = a.G > 1 ? RES_HALO : 0;
  const int j = STEP * w + lc - halo;
  const bool mine = lane < TW && (lc >= 1 || (w == 0 && halo == 0)) &&
                    (lc <= STEP || (w == W - 1 && halo == 0)) && j >= 0 && j < n_own;
  const bool moves = lane >= 1 && lane <= STEP && j > n_lo && j < n_hi - 1 && j < n_own + halo;
  {
    const int jc = j < n_lo ? n_lo : (j >= n_hi ? n_hi - 1 : j);
    if (lane < TW) {
#pragma unroll
      for (int r = 0; r < NC; ++r) cells[w][r][lane] = a.Qin[r * a.pitch + o0 + jc];
    }
  }
  if (threadIdx.x == 0) dead = 0;
  const bool quits = res_quits(a);
  double t = a.t, lmax = 0.0, c[2];
  long long s = 0;
  int to_halo = RES_HALO;
  int bad = 0;
  bool ok = true;
  for (;; ++s) {
    double q[NC];
    auto load = [&]() {
#pragma unroll
      for (int r = 0; r < NC; ++r) q[r] = cells[w][r][lc];
    };
    load();
    int b = 0;
    const double lam = cell_speeds<2, FAST>(mat, q, c, b);
    bad |= mine && b;
    const double m = wave_max_dpp(mine ? lam : 0.0);
    if (lane == 0) red[s & 1][w] = m;
    res_barrier();
    lmax = wave_max_dpp(lane < W ? red[s & 1][lane] : 0.0);
    if (a.G > 1 && w == 0) res_publish(a, s, lmax);
    // face i+1/2 of this lane: its jump as chunk_step tests it
    const double a0n = lane_down(q[0]), a1n = lane_down(q[15]);
    const bool jump = !(((a0n - q[0]) == 0.0) & ((a1n - q[15]) == 0.0)) & (lane < TW - 1) &
                      (j >= n_lo) & (j < n_hi - 1);
    const unsigned long long jumps = __ballot(jump);
    const int faces = __popcll(jumps);
    if (jump) list[w][__popcll(jumps & ((1ull << lane) - 1ull))] = (unsigned char)lane;
    auto wait = [&]() {  // for the team's maximum
      if (a.G == 1) return;
      if (w == 0) {
        double lm = 0.0;
        const bool got = !quits && res_collect<MAXG>(a, s, lm);
        if (lane == 0) {
          team_max = lm;
          if (!got) dead = 1;
        }
      }
      res_barrier();
      lmax = team_max;
      ok = dead == 0;
    };
    // right minus left face flux of every component, without the path terms
    double smin, smax, df[NC];
    int b2 = 0;
    HllCoef hc = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    speed_range2(mat, q, c, smin, smax);
    if constexpr (FLUX == FLUX_RUSANOV) {
      if (a.lxf) {  // the face speed dx / dt
        wait();
        if (!ok) break;
      }
      faces_rusanov2<FAST>(mat, q, smin, smax, a.cfl * rcp(lmax), a.lxf, b2,
                           [&](int r, double d) { df[r] = d; });
    } else {
      double mn, mx;
      mid_range2<FAST>(mat, q, mn, mx);
      hc = hll_coef(mn, mx, smin, lane_down(smax));
      if (lane < TW) {
        bound[w][0][lane] = hc.s_l;
        bound[w][1][lane] = hc.s_r;
        bound[w][2][lane] = hc.isd;
      }
      faces_hll2<FAST>(mat, q, hc, b2, [&](int r, double d, double J) {
        df[r] = d;
        if (jump) path[w][r][lc] = J;
      });
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll 1
    for (int k = lane / GL; k < faces; k += 64 / GL) {
      const int face = list[w][k];
      if constexpr (FLUX == FLUX_RUSANOV)
        face_path2<FAST, GL>(mat, &cells[w][0][0], &path[w][0][0], face, TW, lane & (GL - 1));
      else
        face_path2_hll_lds<FAST, GL>(mat, &cells[w][0][0], &bound[w][0][0], &path[w][0][0], face,
                                     TW, lane & (GL - 1));
    }
    __builtin_amdgcn_wave_barrier();
    if (!(FLUX == FLUX_RUSANOV && a.lxf)) {
      wait();
      if (!ok) break;
    }
    if (s >= a.kmax || !(t < a.t_end)) break;  // main.jl:202 `while t < T`
    const double dtdx = a.cfl * rcp(lmax);
    if (w == 0) {  // the time, by one wave
      const double dt = a.cfl * a.dx / lmax;  // main.jl:212
      if (lane == 0) {
        if (a.dt_hist && a.rank == 0) a.dt_hist[s] = dt;
        tnow[s & 1] = t + dt;
      }
    }
    double upd[NC];
    load();
#pragma unroll
    for (int r = 0; r < NC; ++r) upd[r] = q[r] - dtdx * df[r];
    if (faces) {
#pragma unroll
      for (int r = 0; r < NC; ++r) {
        const double v = jump ? path[w][r][lc] : 0.0;
        double dm = v, dp = v;
        if constexpr (FLUX == FLUX_HLL) {  // the products k_path2_hll stores
          dm = hc.cl * v;
          dp = hc.cr * v;
        }
        upd[r] -= dtdx * (dm + lane_up_z(dp));  // D- of face i+1/2 + D+ of face i-1/2
      }
    }
    if (moves) {
      if (relax > 0.0 || relax_p > 0.0) {
        const double dt = a.cfl * a.dx / lmax;
        if (relax > 0.0) relax_velocity2(mat, upd, exp(-dt * relax));
        if (relax_p > 0.0) relax_pressure2<FAST>(mat, upd, dt * relax_p);
      }
#pragma unroll
      for (int r = 0; r < NC; ++r) cells[w][r][lane] = upd[r];
    }
    const bool renew = a.G > 1 && --to_halo == 0;  // uniform
    if (renew && mine) {
      if (j < RES_HALO) {
#pragma unroll
        for (int r = 0; r < NC; ++r) mine_out[0][j][r] = moves ? upd[r] : q[r];
      }
      if (j >= n_own - RES_HALO) {
#pragma unroll
        for (int r = 0; r < NC; ++r) mine_out[1][j - (n_own - RES_HALO)][r] = moves ? upd[r] : q[r];
      }
    }
    res_barrier();
    t = tnow[s & 1];
    if ((lane == 0 && w > 0) || (lane == TW - 1 && w < W - 1)) {
      const int nb = lane == 0 ? w - 1 : w + 1, nl = lane == 0 ? STEP : 1;
#pragma unroll
      for (int r = 0; r < NC; ++r) cells[w][r][lane] = cells[nb][r][nl];
    }
    if (renew) {
      to_halo = RES_HALO;
      const long long round = (s + 1) / RES_HALO;
      const unsigned tag = a.tag0 + (unsigned)s;
      bool got = true;
      if (w == 0 && a.rank > 0) {
        res_send<NC>(a, round, tag, 0, &mine_out[0][0][0]);
        got = res_receive<NC>(a, round, tag, a.rank - 1, 1, &theirs[0][0][0]);
      }
      if (w == W - 1 && a.rank < a.G - 1) {
        res_send<NC>(a, round, tag, 1, &mine_out[1][0][0]);
        got = res_receive<NC>(a, round, tag, a.rank + 1, 0, &theirs[1][0][0]);
      }
      if (!got) dead = 1;  // seen after the next step's barriers
      res_barrier();
      const bool left = j < 0 && j >= n_lo;
      if (lane < TW && (left || (j >= n_own && j < n_own + RES_HALO && j < n_hi))) {
        const double* e = left ? theirs[0][j + RES_HALO] : theirs[1][j - n_own];
#pragma unroll
        for (int r = 0; r < NC; ++r) cells[w][r][lane] = e[r];
      }
    }
  }
  if (ok) {
    if (mine) {
#pragma unroll
      for (int r = 0; r < NC; ++r) a.Qout[r * a.pitch + o0 + j] = cells[w][r][lc];
      a.Cout[o0 + j] = c[0];
      a.Cout[a.pitch + o0 + j] = c[1];
    }
    if (__any(bad) && lane == 0) atomicOr(a.status, 1);
  }
  return {s, t, lmax, ok};
}

// A material at a wave-uniform address into scalar registers (field by field,
// through the constant address space).
__device__ __forceinline__ MatDev uniform_mat(const MatDev* m) {
  typedef const __attribute__((address_space(4))) MatDev cmat_t;
  cmat_t* g = (cmat_t*)m;
  MatDev d;
  d.rho0 = g->rho0; d.irho0 = g->irho0; d.cv = g->cv; d.t0 = g->t0; d.b0sq = g->b0sq;
  d.k0 = g->k0; d.alpha = g->alpha; d.beta = g->beta; d.gamma = g->gamma;
  d.hk0a2 = g->hk0a2; d.k0_2a = g->k0_2a; d.k0_a = g->k0_a; d.cvt0 = g->cvt0;
  d.icvt0 = g->icvt0; d.hb0sq = g->hb0sq; d.half_a = g->half_a; d.half_b = g->half_b;
  d.half_g = g->half_g; d.ac_t = g->ac_t; d.ac_s = g->ac_s; d.ac_e = g->ac_e;
  d.ac_w = g->ac_w; d.fast = g->fast; d.pad = 0;
  return d;
}

// ---- the time loops of a batch (one phase): a team per problem ---------------

struct BResTeam {  // a problem's team
  long long lo, hi;
  long long slots, border;  // its words in the message buffer
  int G, own;
};
struct BResItem {  // a workgroup's place: rank in the team of a problem
  int p, rank;
};
// Workgroups take the teams' places in the order in which they start, not by
// their block index: whoever waits for a team's missing workgroups then waits
// for the ones that start next, and those find room because every earlier
// team is complete and comes to its end.  Three workgroups share a compute
// unit (one wave of each per SIMD, 168 VGPRs; with two tiles per wave the
// fluxes wait in LDS, 52 KB of it per workgroup), so that one's waits are
// filled by the others: the FP64 units are then busy 0.71 of the time (552 VALU
// instructions per tile and step).  4096 problems of 256 .. 16384 cells, us per
// step, one launch per step against this: Rusanov 780 -> 398, HLL 830 -> 564;
// three tiles per wave at two waves per SIMD: 408 and 582; one tile: 516, 680.
inline constexpr int BRES_BLOCK = 256, BRES_PER_CU = 3;
// Steps of one launch at most.  The first workgroups of a team that is next in
// line wait until an earlier team has taken all its steps, which has to stay
// well below the time after which a wait gives up: a step of a full chip takes
// 9 to 16 us, this many 0.15 to 0.3 s, and a launch more costs 30 us.
inline constexpr long long BRES_STEPS = 1LL << 14;
// This workgroup's problem, and its place in the problem's team (tm's cells and
// messages).
__device__ __forceinline__ int bres_place(int* ticket, const BResItem* items, const BResTeam* teams,
                                          unsigned long long* comm, ResTeam& tm) {
  __shared__ int place;
  if (threadIdx.x == 0) place = atomicAdd(ticket, 1);
  __syncthreads();
  const int item = __builtin_amdgcn_readfirstlane(place);
  const int p = cload(&items[item].p);
  const BResTeam* d = teams + p;
  tm.lo = cload(&d->lo);
  tm.hi = cload(&d->hi);
  tm.G = cload(&d->G);
  tm.rank = cload(&items[item].rank);
  tm.own = cload(&d->own);
  tm.slots = comm + cload(&d->slots);
  tm.border = comm + cload(&d->border);
  return p;
}

// ---- host side --------------------------------------------------------------

// Shape of a team's workgroups: threads, and what a wave holds: tiles of 64
// cells (one phase), or cells (two phases).
struct ResShape {
  int block, tiles;
};
inline constexpr int RES_MAX_TEAM = 256;  // workgroups

// Ticks of the device's 100 MHz counter in a time to wait (0 if it is negative).
inline long long res_ticks(long long microseconds) {
  return std::min(std::max(microseconds, 0LL), 1LL << 40) * 100;
}

// How a problem is laid on the chip (block 0: it is not, and runs step by
// step): the first of these shapes whose team has a compute unit for every
// workgroup.  Fewer waves per SIMD come first, since a step's chain of
// dependent FP64 operations is what a team of few waves waits for (us per
// step, Rusanov / HLL, this shape against the next at the same cells, 59000:
// 4.4 / 3.8 against 4.9 / 4.9; 123000: 5.3 / 5.1 against 7.1 / 8.2; 250000:
// 7.6 / 8.2 against 9.3 / 11.8; the last against one launch per step, 300000:
// 9.5 / 11.8 against 21.1 / 20.3).  Two tiles of 64 cells per wave and three
// fill the registers of two waves per SIMD (200 to 256 VGPRs).
inline constexpr ResShape RES_SHAPES[4] = {{256, 1}, {512, 1}, {512, 2}, {512, 3}};

struct ResPlan {
  ResShape shape;
  int G, own;  // workgroups, and cells of each
};
// The first of `count` shapes (whose single workgroup holds cells_of cells)
// whose team fits.
template <class Cells>
ResPlan res_plan(long long n, int cus, const ResShape* shapes, int count, Cells cells_of) {
  for (int k = 0; k < count; ++k) {
    const int cells = cells_of(shapes[k]), per = cells - 2 * RES_HALO;
    const long long g = n <= cells ? 1 : (n + per - 1) / per;
    if (g <= std::min(cus, RES_MAX_TEAM)) return {shapes[k], (int)g, (int)((n + g - 1) / g)};
  }
  return {{0, 0}, 0, 0};
}
inline ResPlan res_plan1(long long n, int cus) {
  return res_plan(n, cus, RES_SHAPES, 4,
                  [](ResShape s) { return s.block / 64 * s.tiles * TILE + 2; });
}

// 64-bit words of a team's message buffer: slots, then halo words.
inline size_t res_words_of(int G, int nc) {
  return (size_t)2 * G * RES_SLOT + (size_t)2 * G * 2 * RES_HALO * 2 * nc;
}

// Two workgroups on one compute unit would share its SIMDs while other units
// idle: a team's workgroups ask for more LDS than half a unit has.
inline constexpr unsigned RES_ALONE_LDS = 84 * 1024;

template <class Args>
hipError_t res_launch(void (*k)(Args), int block, int G, const Args& a, hipStream_t st) {
  unsigned lds = 0;
  if (G > 1) {
    hipFuncAttributes fa;
    hipError_t e = hipFuncGetAttributes(&fa, (const void*)k);
    if (e == hipSuccess && fa.sharedSizeBytes < RES_ALONE_LDS) {
      lds = RES_ALONE_LDS - (unsigned)fa.sharedSizeBytes;
      e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    }
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k, dim3((unsigned)G), dim3((unsigned)block), lds, st, a);
  return hipGetLastError();
}
// Teams for every problem of a batch (cells [offsets[p], offsets[p + 1])), with
// one tile per wave or two.  One has the shorter chain of work per step and
// wastes less of a short problem's last wave, two need fewer exchanges and, the
// chip full, 1.27 times less time per tile (516 against 398 us above).  So one
// when all its workgroups are on the chip at once (64 problems of 100 .. 3000
// cells: 3.7 against 5.0 us per step) or when its tiles are that many fewer
// (1000 of 60 .. 700 cells: 12.5 against 14.5), else two, the largest problems
// first.  tiles = 0 if a problem does not fit, or if a launch per step is faster
// (bres_pays).
struct BResPlan {
  int tiles = 0;
  bool waits = false;  // some problem has more than one workgroup
  std::vector<BResTeam> teams;
  std::vector<BResItem> items;
  // 64-bit words of the message buffer: the ticket counter and all slots (to be
  // cleared before a launch), then the halo words
  size_t clear = 0, words = 0;
};
// Many problems of a few cells: a workgroup's four waves all work, however few
// cells its problem has, where a launch per step takes a wave per tile.  So once
// the chip is full, one launch for all steps pays only if it takes less time than
// a launch per step; both by us per step as measured on 256 compute units (the
// latter in a captured graph, its capture and launch included), in the order
// Rusanov, HLL, then with general exponents.  A launch per step against this,
// us per step: 16384 problems of 3 cells 43 and 71 (HLL 45 and 106), of 62 cells
// 57 and 71 (58 and 106), of 100 cells 94 and 71 (102 and 106), of 124 cells 110
// and 72 (114 and 106); 4096 of 3 cells 15 and 18, of 62 cells 20 and 18 (19 and
// 27); 2048 of 3 cells 11 and 10 (12 and 14), of 62 cells 17 and 10 (18 and 14).
inline bool bres_pays(long long groups, int tiles_per_wave, long long tiles, long long cells,
                      int cus, bool hll, bool fast) {
  if (groups <= (long long)BRES_PER_CU * cus) return true;
  constexpr double group_ns[4][2] = {{4.5, 7.9}, {6.45, 11.7}, {5.5, 10.1}, {8.65, 15.9}};
  constexpr double step[4] = {1.0, 1.04, 1.10, 1.22};
  const int k = (hll ? 1 : 0) + (fast ? 0 : 2);
  const double once = 0.8 + 1e-3 * group_ns[k][tiles_per_wave - 1] * (double)groups;
  const double each = step[k] * (8.0 + 2.1e-3 * (double)tiles + 15.5e-6 * (double)cells);
  return once <= each;
}
inline BResPlan bres_plan(const std::vector<long long>& offsets, int cus, int nc, bool hll, bool fast) {
  const int P = (int)offsets.size() - 1;
  BResPlan pl;
  pl.teams.resize(P);
  auto fit = [&](int t) -> long long {  // workgroups with t tiles per wave
    const long long one = BRES_BLOCK / 64 * t * TILE + 2, per = one - 2 * RES_HALO;
    long long groups = 0;
    pl.waits = false;
    for (int p = 0; p < P; ++p) {
      const long long n = offsets[p + 1] - offsets[p];
      const long long g = n <= one ? 1 : (n + per - 1) / per;
      if (g > std::min(cus, RES_MAX_TEAM)) return -1;
      pl.teams[p] = {offsets[p], offsets[p + 1], 0, 0, (int)g, (int)((n + g - 1) / g)};
      pl.waits = pl.waits || g > 1;
      groups += g;
    }
    return groups;
  };
  const long long groups2 = fit(2), groups1 = fit(1);
  const bool one = groups1 >= 0 && (groups1 <= BRES_PER_CU * cus || 1.27 * groups1 < 2.0 * groups2);
  const long long groups = one ? groups1 : fit(2);
  if (groups < 0 || groups > 0x7fffffffLL) return pl;
  long long tiles = 0;
  for (int p = 0; p < P; ++p) tiles += (offsets[p + 1] - offsets[p] + TILE - 1) / TILE;
  if (!bres_pays(groups, one ? 1 : 2, tiles, offsets[P] - offsets[0], cus, hll, fast)) return pl;
  std::vector<int> order(P);
  for (int p = 0; p < P; ++p) order[p] = p;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
    return pl.teams[x].hi - pl.teams[x].lo > pl.teams[y].hi - pl.teams[y].lo;
  });
  pl.items.reserve((size_t)groups);
  size_t at = 1;  // after the ticket counter
  for (int p : order) {
    BResTeam& t = pl.teams[p];
    for (int r = 0; r < t.G; ++r) pl.items.push_back({p, r});
    t.slots = (long long)at;
    if (t.G > 1) at += (size_t)2 * t.G * RES_SLOT;
  }
  pl.clear = at;
  for (int p : order) {
    BResTeam& t = pl.teams[p];
    t.border = (long long)at;
    if (t.G > 1) at += (size_t)2 * t.G * 2 * RES_HALO * 2 * nc;
  }
  pl.words = at;
  pl.tiles = one ? 1 : 2;
  return pl;
}

}  // namespace hes
