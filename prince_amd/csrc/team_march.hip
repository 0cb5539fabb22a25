// team_march.hip -- the whole redshift march of a shared-schedule batch in one
// cooperative launch (gfx950).
//
// What bounds the march when every stage is its own kernel: a stage moves
// 3 MB of coupling values and the state, about 1 us of traffic for one
// right-hand side, but costs two launches and their dependency gaps (11.9 us
// per stage at K = 1, 33 us at K = 64), and it reads the same coupling values
// again in each of the ~20 stages of a refresh window.  Here the chip is cut
// into teams of workgroups, one workgroup per CU; a team owns a share of the
// right-hand sides for the whole march (columns never exchange data), and a
// workgroup of it owns species rows whose coupling values of the current
// window stay in its LDS (93 KB per CU for the A <= 56 run on a 32-CU team).
// Between stages only the state crosses workgroups: x and a are stored and
// loaded with agent-scope cache policy (sc1), so no cache write-back or
// invalidation is needed, and a team barrier costs 1.5 us (32 workgroups of
// one XCD) to 2.6 us (256).  A full agent-scope release / acquire pair instead
// measured 37 us per stage: it writes back and invalidates the whole L2.
// Measured per stage of the A <= 56 run, stage kernels -> march: K = 1 11.5 ->
// 6.3 us, K = 7 20 -> 6.8, K = 64 33 -> 16.5, K = 300 129 -> 45, K = 512 92 -> 79;
// two fields, K = 48: 48 -> 21.6.  What bounds it, by counters: K = 1 a serial chain
// (the SIMDs issue 0.6 of 6.2 us, waves wait 70 % of their time: barrier, load
// latency, one row's instructions); K = 64 the same at 8 us of issue per SIMD, 77 %
// of the L2 requests hit and 33 MB go past the L2 per stage; K = 512 traffic: a team's
// state is 10 MB per array against 4 MB of L2, 40 % of the requests miss and 373 MB
// per stage pass at 4.7 TB/s, the rate of a large copy.  With few rows or beyond
// those columns the stage kernels are faster (solvers/team.py, march_pays).
//
// Teams are workgroups blockIdx % nteam, which the dispatcher places on one
// XCD (nteam = 8) or on a pair of XCDs (nteam = 4); only speed depends on that
// placement, the sc1 accesses are coherent over the whole device.
//
// Dense rows (protons: one band block from almost every species; He-4: one
// diagonal block from almost every species) would be one workgroup's serial
// chain.  No nucleus feeds a heavier one, so the heavy rows never read the
// dense rows or the few light rows that read those ("tail" rows), and the tail
// runs one phase behind: in the phase of stage p the heavy rows do stage p,
// `ndwg` workgroups sum the dense rows' blocks over the heavy mothers (shared
// out by mothers, a mother panel loaded once for both rows), and `nfwg`
// workgroups finish the tail rows of stage p - 1 from the partials of the
// phase before.  One barrier per stage then orders everything; finishing the
// dense rows inside the stage behind a second barrier measured 7.0 us per stage
// at K = 1.
//
// Lanes: a wave holds two right-hand sides, 32 lanes each, two energy bins per
// lane, so every state and value access is 16 bytes per lane.  8-byte loads of
// the same panels stop at 18.8 TB/s over the chip (half of a CU's load path),
// 16-byte ones reach 28 - 32 TB/s with sc1 and 31 - 36 without, where the panels
// fit an L2; a shift by one bin also moves half as many registers.
//
// Every wait is bounded: a workgroup that polls SPIN_LIMIT times (prh_team.spin_limit)
// without progress raises the abort word and leaves, and the others do when they
// next wait.  Which of them still stored results is then a matter of timing, so a
// launch behind the march reads the word and, where it is raised, fills with NaN
// everything that march writes for its caller: no result of an aborted march, nor
// of what follows from it, is finite.  Within a process marches of one device run one
// after the other (march_launch.h).  Those of two processes on one card meet only in
// the driver's scheduling of cooperative launches, which was not measured.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../../include/prince_hip.h"
#include "internal.h"
#include "march_launch.h"

namespace {

#include "stage_math.h"

constexpr int TWAVES = 16;  // waves per workgroup (128 registers each)
constexpr int TTHREADS = TWAVES * WAVE;
constexpr int TDENSE = 2;   // dense rows per operator
constexpr int TSUMS = 3;    // sums a dense-row workgroup may form: those rows, and the EM weights
constexpr int TCONST = 9;   // LDS rows: 7 FD coefficients, energy grid, FD diagonal
constexpr int SC1 = 16;     // buffer cache policy: agent scope
constexpr int SPIN_LIMIT = 1 << 25;
// sync words (32-bit) of prh_team::sync: per team, 64 words apart
constexpr int SY_SUB = 0;       // [8 teams][8 sub-groups] arrival counters
constexpr int SY_ROOT = 4096;   // [8 teams] arrivals of complete sub-groups
constexpr int SY_ABORT = 4608;
constexpr int SY_WORDS = 4672;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));  // bins 2 l, 2 l + 1 of lane l of a half

// state access: agent scope for x, a and the partials, plain for F(x) (read back
// by the wave that wrote it)
template <int POLICY>
__device__ __forceinline__ d2 pload(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, POLICY));
}
template <int POLICY>
__device__ __forceinline__ void pstore(d2 v, __amdgpu_buffer_rsrc_t r, int voff, int soff) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voff, soff, POLICY);
}

// The arguments stay in the kernel's argument segment and are read from there,
// phase by phase, through the scalar cache: as ordinary by-value arguments the
// compiler keeps some 60 pointers in registers over the whole march and spills
// (300 register moves to and from lanes of vector registers per phase).
struct TeamArgs {
  prh_operator op;
  prh_schedule sch;
  prh_state st;
  prh_team tm;
  int k_begin, k_end;
};
#define CONST_SPACE const __attribute__((address_space(4)))
typedef CONST_SPACE TeamArgs CArgs;
typedef CONST_SPACE prh_operator COp;
typedef CONST_SPACE prh_schedule CSch;
typedef CONST_SPACE prh_state CSt;
typedef CONST_SPACE prh_team CTm;
// the same pointer, as far as the compiler knows another one: what was read
// through it before is read again
__device__ __forceinline__ CArgs* reread(CArgs* a) {
  asm volatile("" : "+s"(a));
  return a;
}

// Read-only tables at wave-uniform indices: constant-space loads go through the
// scalar cache, where a plain load becomes a vector load (the compiler cannot
// rule out that the march's stores change them) and a 0.3 us wait in a chain.
template <typename V>
__device__ __forceinline__ V cload(const V* p) {
  return *reinterpret_cast<CONST_SPACE V*>(reinterpret_cast<uintptr_t>(p));
}

// This lane's place in the wave.
struct Lane {
  int id;           // 0 .. 63
  int half;         // right-hand side of the pair
  int bin;          // first of its two bins
  int off;          // byte offset of its bins in the pair's [2][64] panel
  bool first, last; // bins 0, 1 / 62, 63
};
__device__ __forceinline__ Lane lane_of() {
  Lane n;
  n.id = threadIdx.x & (WAVE - 1);
  n.half = n.id >> 5;
  n.bin = 2 * (n.id & 31);
  n.off = n.id * 16;
  n.first = n.bin == 0;
  n.last = n.bin == 62;
  return n;
}

// Lane shifts inside a half: the neighbour lane's value, zero past the ends (the
// other half is another right-hand side).
__device__ __forceinline__ double prev1(const Lane& n, double v) {
  const double r = lane_prev(v);
  return n.first ? 0.0 : r;
}
__device__ __forceinline__ double next1(const Lane& n, double v) {
  const double r = lane_next(v);
  return n.last ? 0.0 : r;
}
// the panel moved down by one bin: bin i receives bin i + 1
__device__ __forceinline__ d2 shift_bin(const Lane& n, d2 v) {
  const double t = next1(n, v.x);
  return d2{v.y, t};
}

struct TeamLds {
  double* cst;  // [9][64]
  double* rp;   // [2][fields][64] pair-production rate of the window
  double* red;  // [16 waves][2][64 lanes][2] partial sums of the dense rows' mother groups
  double* coef; // [2][coefs] source coefficients of the team's columns, this step's
                // and the next one's
  double* val;  // [fields][slots][64] coupling values of the window (finishing
                // workgroups: two such sets, they also need the window before)
  int slots, coefs;
};
__device__ __forceinline__ d2 lds2(const double* base, int slot, int bin) {
  return *reinterpret_cast<const d2*>(base + slot * WAVE + bin);
}

struct StepIn {
  int step, ridx;  // ridx: slot of the record arrays, -1 when not recorded
  double dl, h, hadia, finj;
};
// Per row: pair-production scale and source slot (-1: none).
struct RowConst {
  double pscale;
  int sslot;
};
__device__ __forceinline__ RowConst row_const(COp& op, int da) {
  return RowConst{cload(op.pscale + da),
                  (op.flags & PRH_F_INJECTION) ? cload(op.src_slot + da) : -1};
}

// The state arrays as buffers over their whole [nspec][K][64] extent (one
// descriptor each): row, column and panel offsets are scalar byte offsets.
struct TeamState {
  __amdgpu_buffer_rsrc_t x, a, f;
  __amdgpu_buffer_rsrc_t part;  // [2 stages][nparts][K][64] partial sums of the tail rows
  int pb;                       // bytes of one species' [K][64] panel
  int phalf;                    // bytes of one stage's partials
};

// Source coefficients norm evolution(z) of a step for the team's nc columns from c0:
// read a step ahead into a register by coef_ahead, into LDS by coef_stage after
// the step's work, so that no stage waits for memory it never touched before (about
// 2 us; 5 us per stage on the rows with sources at K = 64).
__device__ __forceinline__ double coef_ahead(COp& op, CSch& sch, int step, int c0, int nc) {
  const int J = op.nsrc;
  if (!(op.flags & PRH_F_INJECTION) || J < 1) return 0.0;  // uniform
  const int i = (int)threadIdx.x < J * nc ? threadIdx.x : J * nc - 1;
  const int j = i / nc;
  return sch.src_coef[((int64_t)step * J + j) * op.K + c0 + (i - j * nc)];
}
__device__ __forceinline__ void coef_stage(const TeamLds& L, int step, double c) {
  if ((int)threadIdx.x < L.coefs) L.coef[(step & 1) * L.coefs + threadIdx.x] = c;
}

// Source sums sum_j norm evolution(z) g_j of source slot sslot for the pairs from k0.
template <int KP>
__device__ __forceinline__ void team_source(COp& op, const TeamLds& L, int step,
                                            int sslot, int c0, int k0, int kend, const Lane& n,
                                            d2 (&src)[KP]) {
  if (sslot < 0) return;
  const int J = op.nsrc, K = op.K, nc = kend - c0;
  for (int j = 0; j < J; ++j) {
    d2 g[KP];
    double c[KP];
#pragma unroll
    for (int p = 0; p < KP; ++p) {
      const int kk = k0 + 2 * p + n.half;
      const int k = kk < kend ? kk : kend - 1;
      g[p] = *reinterpret_cast<const d2*>(op.src_grid +
                                          (((int64_t)sslot * J + j) * K + k) * WAVE + n.bin);
      c[p] = L.coef[(step & 1) * L.coefs + j * nc + k - c0];
    }
#pragma unroll
    for (int p = 0; p < KP; ++p) src[p] = (j == 0) ? c[p] * g[p] : src[p] + c[p] * g[p];
  }
}

// Diagonal factors of one bin in stage s2 (propagation.py:1389-1422,
// etd2.py:329-390).
__device__ __forceinline__ void bin_factors(int s2, double kadia, double pscale, double rate,
                                            double mdiag, double ddiag, double dl, double h,
                                            bool pdiff, double& kap, double& e, double& phi) {
  kap = kadia + pscale * rate;
  double dval = mdiag * dl;
  if (pdiff) {
    double kxd = kap * ddiag;
    kxd = kxd * dl;
    dval = dval + kxd;
  }
  const double hd = dval * h;
  e = exp(hd);
  phi = s2 ? phi2_of(hd, e) : phi1_of(hd, e);
}

// Factors of a row for one pair of right-hand sides.  One-field operators have the
// same for every pair: computed once, each half of the wave one of the two bins
// (half the exponentials), then exchanged.
struct RowFactors {
  d2 kap, e, phi;
};
// {lane l's value, lane l + 32's value} in both halves (v_permlane32_swap: no LDS)
__device__ __forceinline__ d2 from_halves(double v) {
  const u32x2 b = __builtin_bit_cast(u32x2, v);
  const auto lo = __builtin_amdgcn_permlane32_swap(b.x, b.x, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(b.y, b.y, false, false);
  return d2{__builtin_bit_cast(double, u32x2{lo[0], hi[0]}),
            __builtin_bit_cast(double, u32x2{lo[1], hi[1]})};
}
template <bool TWO>
__device__ __forceinline__ RowFactors row_factors(COp& op, const TeamLds& L,
                                                  const StepIn& si, int s2, double pscale, int slot,
                                                  int k, const Lane& n) {
  const bool pdiff = (op.flags & PRH_F_PARTIAL_DIFF) != 0;
  RowFactors f;
  if constexpr (!TWO) {
    const int bin = n.bin + n.half;
    double kap, e, phi;
    bin_factors(s2, si.hadia * L.cst[7 * WAVE + bin], pscale, L.rp[bin], L.val[slot * WAVE + bin],
                L.cst[8 * WAVE + bin], si.dl, si.h, pdiff, kap, e, phi);
    f.kap = from_halves(kap);
    f.e = from_halves(e);
    f.phi = from_halves(phi);
  } else {
    const double s = op.escale[k];
#pragma unroll 1
    for (int i = 0; i < 2; ++i) {
      const int bin = n.bin + i;
      double kap, e, phi;
      bin_factors(s2, si.hadia * L.cst[7 * WAVE + bin], pscale, L.rp[bin] + s * L.rp[WAVE + bin],
                  L.val[slot * WAVE + bin] + s * L.val[(L.slots + slot) * WAVE + bin],
                  L.cst[8 * WAVE + bin], si.dl, si.h, pdiff, kap, e, phi);
      if (i == 0) {
        f.kap.x = kap;
        f.e.x = e;
        f.phi.x = phi;
      } else {
        f.kap.y = kap;
        f.e.y = e;
        f.phi.y = phi;
      }
    }
  }
  return f;
}

// Epilogue of row da for the pairs of right-hand sides from k0 (below kend): the
// same expressions per bin as the per-stage kernels' epilogue.
template <int KP, bool TWO, bool REC>
__device__ __forceinline__ void team_epilogue(COp& op, CSt& st,
                                              const TeamState& T, const TeamLds& L,
                                              const StepIn& si, int s2, const RowFactors& f0,
                                              const RowConst& rc, int da, int slot, int k0,
                                              int kend, const Lane& n, const d2 (&acc)[KP],
                                              const d2 (&xo)[KP], const d2 (&fo)[KP],
                                              const d2 (&src)[KP]) {
  const bool pdiff = (op.flags & PRH_F_PARTIAL_DIFF) != 0;
#pragma unroll
  for (int p = 0; p < KP; ++p) {
    const int kp = k0 + 2 * p;
    if (kp >= kend) break;  // uniform over the wave
    const int k = kp + n.half;
    RowFactors f = f0;
    if (TWO) f = row_factors<true>(op, L, si, s2, rc.pscale, slot, k < kend ? k : kend - 1, n);
    d2 out = acc[p];
    if (pdiff) {
      const d2 kx = f.kap * xo[p];
      // stencil neighbours of bins 2 l and 2 l + 1, added in the order -3 .. 3.
      // Past the ends of a half the shifts bring the other column's bins, which
      // meet coefficients that are exactly zero; masked unless all are finite
      // (K = 64 33.3 -> 32.7 ms per 2000 stages with the masks off).
      double m1 = lane_prev(kx.y);  // bin 2 l - 1
      double m2 = lane_prev(kx.x);  // bin 2 l - 2
      double m3 = lane_prev(m1);    // bin 2 l - 3
      double q2 = lane_next(kx.x);  // bin 2 l + 2
      double q3 = lane_next(kx.y);  // bin 2 l + 3
      double q4 = lane_next(q2);    // bin 2 l + 4
      if (__builtin_expect(!__all(isfinite(kx.x) && isfinite(kx.y)), 0)) {
        m1 = n.first ? 0.0 : m1;
        m2 = n.first ? 0.0 : m2;
        m3 = n.bin < 4 ? 0.0 : m3;
        q2 = n.last ? 0.0 : q2;
        q3 = n.last ? 0.0 : q3;
        q4 = n.bin > 59 ? 0.0 : q4;
      }
      d2 dx = {0.0, 0.0};
      dx += lds2(L.cst, 0, n.bin) * d2{m3, m2};
      dx += lds2(L.cst, 1, n.bin) * d2{m2, m1};
      dx += lds2(L.cst, 2, n.bin) * d2{m1, kx.x};
      dx += lds2(L.cst, 4, n.bin) * d2{kx.y, q2};
      dx += lds2(L.cst, 5, n.bin) * d2{q2, q3};
      dx += lds2(L.cst, 6, n.bin) * d2{q3, q4};
      out = out + dx;
    }
    out = out * si.dl;
    if (rc.sslot >= 0) out = out + si.finj * src[p];
    if (k >= kend) continue;  // the odd last right-hand side's idle half
    const int co = da * T.pb + kp * (WAVE * 8);
    const int64_t nk = (int64_t)op.nspec * op.K * WAVE;
    const int64_t rec = REC ? si.ridx * nk + ((int64_t)da * op.K + k) * WAVE + n.bin : 0;
    if (s2 == 0) {
      d2 a = f.e * xo[p];
      d2 sc = f.phi * out;
      sc = sc * si.h;
      a = a + sc;
      pstore<SC1>(a, T.a, n.off, co);
      pstore<0>(out, T.f, n.off, co);
      if (REC && si.ridx >= 0) {
        *reinterpret_cast<d2*>(st.rec_x + rec) = xo[p];
        *reinterpret_cast<d2*>(st.rec_a + rec) = a;
        *reinterpret_cast<d2*>(st.rec_fx + rec) = out;
      }
    } else {
      d2 sc = out - fo[p];
      sc = sc * si.h;
      sc = sc * f.phi;
      pstore<SC1>(xo[p] + sc, T.x, n.off, co);
      if (REC && si.ridx >= 0) *reinterpret_cast<d2*>(st.rec_fa + rec) = out;
    }
  }
}

// A wave's rows: row a, or two rows a and b (b < 0: none) read with one walk over
// their mothers, so that a panel both rows read is loaded once (1.4 blocks per
// panel on the A <= 56 run).  Lane e holds entry e (mother, LDS slot of the block):
// first the n2 mothers of both rows (slot: row a's block, slot + 1 row b's), then
// na of row a alone, then nb of row b alone.  part >= 0: a tail row whose coupling
// sum over the heavy mothers goes to the partial buffer at that byte offset.
struct RowTask {
  int a, b, n2, na, nb, diag_a, diag_b, part_a, part_b;
  RowConst ca, cb;
  int mo, sl;  // lane entries
};

// Own state (and, in stage 2, F(x)) of row da for the pairs from k0.
template <int KP>
__device__ __forceinline__ void own_loads(const TeamState& T, int s2, int da, int k0, const Lane& n,
                                          d2 (&xo)[KP], d2 (&fo)[KP]) {
  const auto y = s2 ? T.a : T.x;
#pragma unroll
  for (int p = 0; p < KP; ++p) {
    const int so = da * T.pb + (k0 + 2 * p) * (WAVE * 8);
    xo[p] = pload<SC1>(y, n.off, so);
    fo[p] = pload<0>(T.f, n.off, so);  // stage 1 does not use it
  }
}

// Coupling of U entries from e on: both rows' blocks (BOTH) or those of one row.
// Straight-line: U x KP panel loads, the values from LDS, then the products.
template <int U, int KP, bool TWO, bool BOTH>
__device__ __forceinline__ void couple_chunk(const TeamState& T, const TeamLds& L,
                                             __amdgpu_buffer_rsrc_t y, const RowTask& rt, int e,
                                             int cb, const Lane& n, d2 (&accA)[KP], d2 (&accB)[KP],
                                             d2 (&accAE)[KP], d2 (&accBE)[KP]) {
  d2 xv[U][KP], ma[U], mb[U], mae[U], mbe[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int po = __builtin_amdgcn_readlane(rt.mo, e + u) * T.pb + cb;
#pragma unroll
    for (int p = 0; p < KP; ++p) xv[u][p] = pload<SC1>(y, n.off, po + p * (2 * WAVE * 8));
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int sl = __builtin_amdgcn_readlane(rt.sl, e + u);
    ma[u] = lds2(L.val, sl, n.bin);
    if (BOTH) mb[u] = lds2(L.val, sl + 1, n.bin);
    if (TWO) {
      mae[u] = lds2(L.val, L.slots + sl, n.bin);
      if (BOTH) mbe[u] = lds2(L.val, L.slots + sl + 1, n.bin);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int p = 0; p < KP; ++p) {
      accA[p] += ma[u] * xv[u][p];
      if (BOTH) accB[p] += mb[u] * xv[u][p];
      if (TWO) {
        accAE[p] += mae[u] * xv[u][p];
        if (BOTH) accBE[p] += mbe[u] * xv[u][p];
      }
    }
  }
}
// Entries [e, e + m): chunks of U, then what is left in powers of two.
template <int U, int KP, bool TWO, bool BOTH>
__device__ __forceinline__ void couple_run(const TeamState& T, const TeamLds& L,
                                           __amdgpu_buffer_rsrc_t y, const RowTask& rt, int e, int m,
                                           int cb, const Lane& n, d2 (&accA)[KP], d2 (&accB)[KP],
                                           d2 (&accAE)[KP], d2 (&accBE)[KP]) {
#pragma unroll 1
  for (; m >= U; m -= U, e += U)
    couple_chunk<U, KP, TWO, BOTH>(T, L, y, rt, e, cb, n, accA, accB, accAE, accBE);
  if (U > 2 && (m & 2)) {
    couple_chunk<2, KP, TWO, BOTH>(T, L, y, rt, e, cb, n, accA, accB, accAE, accBE);
    e += 2;
  }
  if (m & 1) couple_chunk<1, KP, TWO, BOTH>(T, L, y, rt, e, cb, n, accA, accB, accAE, accBE);
}

// One stage of a row task for the KP pairs of right-hand sides from k0.  Pairs
// past kend read other panels, or zeros past the array, and are not stored: on gfx950
// the range check of a buffer load takes the scalar offset in, also one beyond the
// range (checked with a descriptor shorter than its allocation).  Clamping the
// columns instead cost 3.7 % at K = 64.
template <int KP, bool TWO, bool REC>
__device__ __forceinline__ void team_rows(COp& op, CSch& sch,
                                          CSt& st, const TeamState& T,
                                          const TeamLds& L, const StepIn& si, int s2,
                                          const RowTask& rt, const RowFactors& fa,
                                          const RowFactors& fb, int c0, int k0, int kend,
                                          const Lane& n) {
  constexpr int U = TWO ? 2 : 4;
  const auto y = s2 ? T.a : T.x;
  d2 acc[2][KP], accE[2][KP], xo[KP], fo[KP];
#pragma unroll
  for (int p = 0; p < KP; ++p)
    acc[0][p] = acc[1][p] = accE[0][p] = accE[1][p] = d2{0.0, 0.0};
  const int cb = k0 * (WAVE * 8);
  couple_run<U, KP, TWO, true>(T, L, y, rt, 0, rt.n2, cb, n, acc[0], acc[1], accE[0], accE[1]);
  couple_run<U, KP, TWO, false>(T, L, y, rt, rt.n2, rt.na, cb, n, acc[0], acc[0], accE[0], accE[0]);
  couple_run<U, KP, TWO, false>(T, L, y, rt, rt.n2 + rt.na, rt.nb, cb, n, acc[1], acc[1], accE[1],
                                accE[1]);
  if (TWO) {
#pragma unroll
    for (int p = 0; p < KP; ++p) {
      const int k = k0 + 2 * p + n.half;
      const double s = op.escale[k < kend ? k : kend - 1];
      acc[0][p] = acc[0][p] + s * accE[0][p];
      acc[1][p] = acc[1][p] + s * accE[1][p];
    }
  }
  // the two rows' ends as a loop: half the code in the instruction cache
  RowFactors f0 = fa;
  RowConst rc = rt.ca;
  int da = rt.a, diag = rt.diag_a, part = rt.part_a;
#pragma unroll 1
  for (int r = 0;;) {
    if (part >= 0) {
#pragma unroll
      for (int p = 0; p < KP; ++p)
        if (k0 + 2 * p + n.half < kend)
          pstore<SC1>(acc[0][p], T.part, n.off,
                      part + (s2 ? T.phalf : 0) + (k0 + 2 * p) * (WAVE * 8));
    } else {
      own_loads<KP>(T, s2, da, k0, n, xo, fo);
      d2 src[KP];
#pragma unroll
      for (int p = 0; p < KP; ++p) src[p] = d2{0.0, 0.0};
      team_source<KP>(op, L, si.step, rc.sslot, c0, k0, kend, n, src);
      team_epilogue<KP, TWO, REC>(op, st, T, L, si, s2, f0, rc, da, diag, k0, kend, n, acc[0], xo,
                                  fo, src);
    }
    if (++r == 2 || rt.b < 0) break;
    f0 = fb;
    rc = rt.cb;
    da = rt.b;
    diag = rt.diag_b;
    part = rt.part_b;
#pragma unroll
    for (int p = 0; p < KP; ++p) acc[0][p] = acc[1][p];
  }
}

// The same for one row and one pair of right-hand sides (teams of one or two
// columns), ordered for latency: every load is issued first, the diagonal
// factors are computed while they travel.  SPLIT (one right-hand side): the
// upper half of the wave takes every second mother instead of a second column.
template <bool TWO, bool REC, bool SPLIT>
__device__ __forceinline__ void team_row1(COp& op, CSch& sch,
                                          CSt& st, const TeamState& T,
                                          const TeamLds& L, const StepIn& si, int s2,
                                          const RowTask& rt, int k0, int kend, const Lane& n) {
  constexpr int U = SPLIT ? 8 : 12;
  constexpr int NB = SPLIT ? 2 : 1;  // mothers per load
  const auto y = s2 ? T.a : T.x;
  const int cb = k0 * (WAVE * 8);
  const d2 z = {0.0, 0.0};
  d2 acc[1] = {z}, xo[1] = {z}, fo[1] = {z}, src[1] = {z}, accE = z;
  RowFactors f0{};
  // offset of entry e's panel for this lane (SPLIT: e or e + 1 by half)
  auto panel = [&](int e, int& slot, bool& has) {
    int po = __builtin_amdgcn_readlane(rt.mo, e) * T.pb;
    slot = __builtin_amdgcn_readlane(rt.sl, e);
    has = true;
    if (SPLIT) {
      const int e1 = e + 1 < rt.na ? e + 1 : e;
      const int p1 = __builtin_amdgcn_readlane(rt.mo, e1) * T.pb;
      const int s1 = __builtin_amdgcn_readlane(rt.sl, e1);
      po = n.half ? p1 : po;
      slot = n.half ? s1 : slot;
      has = e + n.half < rt.na;
    }
    return po;
  };
  for (int e = 0;; e += U * NB) {
    d2 xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (e + u * NB < rt.na) {
        int slot;
        bool has;
        const int po = panel(e + u * NB, slot, has);
        xv[u] = SPLIT ? pload<SC1>(y, n.bin * 8 + po, cb) : pload<SC1>(y, n.off, po + cb);
      }
    }
    if (e == 0 && rt.part_a < 0) {
      own_loads<1>(T, s2, rt.a, k0, n, xo, fo);
      team_source<1>(op, L, si.step, rt.ca.sslot, k0, k0, kend, n, src);
      if (!TWO) f0 = row_factors<false>(op, L, si, s2, rt.ca.pscale, rt.diag_a, k0, n);
    }
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += 4) {
      d2 mc[4], me[4];
      bool has[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int slot;
        const int ee = e + (u0 + u) * NB;
        panel(ee < rt.na ? ee : rt.na - 1 < 0 ? 0 : rt.na - 1, slot, has[u]);
        mc[u] = lds2(L.val, slot, n.bin);
        if (TWO) me[u] = lds2(L.val, L.slots + slot, n.bin);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (e + (u0 + u) * NB < rt.na) {
          // a half without a block adds 0 * 0, whatever the panel holds
          const d2 x = has[u] ? xv[u0 + u] : z;
          acc[0] += mc[u] * x;
          if (TWO) accE += me[u] * x;
        }
      }
    }
    if (e + U * NB >= rt.na) break;
  }
  if (TWO) {
    const int k = k0 + (SPLIT ? 0 : n.half);
    acc[0] = acc[0] + op.escale[k < kend ? k : kend - 1] * accE;
  }
  if (SPLIT) {
    const d2 sx = from_halves(acc[0].x), sy = from_halves(acc[0].y);
    acc[0] = d2{sx.x + sx.y, sy.x + sy.y};
  }
  if (rt.part_a >= 0) {
    if (k0 + n.half < kend)
      pstore<SC1>(acc[0], T.part, n.off, rt.part_a + (s2 ? T.phalf : 0) + cb);
    return;
  }
  team_epilogue<1, TWO, REC>(op, st, T, L, si, s2, f0, rt.ca, rt.a, rt.diag_a, k0, kend, n, acc, xo,
                             fo, src);
}

// A tail row to finish; its blocks from tail mothers sit one per lane.
struct FinTask {
  int da, slot, p0, pstep, pn, nb;
  RowConst rc;
  int mo, sl, band;  // lane entries: mother, LDS slot, first diagonal | diagonals << 8
};
__device__ __forceinline__ FinTask fin_task(COp& op, CTm& tm, int f,
                                            int lane) {
  const int* fr = tm.fin + 8 * f;
  FinTask r;
  r.da = cload(fr);
  r.slot = cload(fr + 1);
  r.p0 = cload(fr + 2);
  r.pstep = cload(fr + 3);
  r.pn = cload(fr + 4);
  r.nb = cload(fr + 6);
  r.rc = row_const(op, r.da);
  r.mo = r.sl = r.band = 0;
  if (lane < r.nb) {
    const int* q = tm.fin_blk + 4 * (cload(fr + 5) + lane);
    r.mo = q[0];
    r.sl = q[1];
    r.band = q[2] | q[3] << 8;
  }
  return r;
}

// One stage of a tail row for the pair of right-hand sides from k0: the partial
// sums of its heavy mothers (of this stage) in their order, then its blocks from
// tail mothers.  Every load is issued before the first use.
template <bool TWO, bool REC>
__device__ __forceinline__ void team_finish(COp& op, CSch& sch,
                                            CSt& st, const TeamState& T,
                                            const TeamLds& L, const StepIn& si, int stage,
                                            const FinTask& ft, int c0, int k0, int kend,
                                            const Lane& n) {
  constexpr int U = 6, UB = 5;
  const auto y = stage ? T.a : T.x;
  const int pbase = stage ? T.phalf : 0;
  const int cb = k0 * (WAVE * 8);
  const d2 z = {0.0, 0.0};
  d2 acc[1] = {z}, xo[1], fo[1], src[1] = {z};
  d2 accB = z, accE = z, xv[UB], pv[U];
#pragma unroll
  for (int u = 0; u < UB; ++u)
    if (u < ft.nb) xv[u] = pload<SC1>(y, n.off, __builtin_amdgcn_readlane(ft.mo, u) * T.pb + cb);
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u < ft.pn) pv[u] = pload<SC1>(T.part, n.off, pbase + (ft.p0 + u * ft.pstep) * T.pb + cb);
  own_loads<1>(T, stage, ft.da, k0, n, xo, fo);
  team_source<1>(op, L, si.step, ft.rc.sslot, c0, k0, kend, n, src);
  // one part after the other: all of them in flight at once would spill
  __builtin_amdgcn_sched_barrier(0);
  for (int g = 0;;) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (g + u < ft.pn) acc[0] += pv[u];
    g += U;
    if (g >= ft.pn) break;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (g + u < ft.pn)
        pv[u] = pload<SC1>(T.part, n.off, pbase + (ft.p0 + (g + u) * ft.pstep) * T.pb + cb);
  }
  __builtin_amdgcn_sched_barrier(0);
  RowFactors f0{};
  if (!TWO) f0 = row_factors<false>(op, L, si, stage, ft.rc.pscale, ft.slot, k0, n);
  __builtin_amdgcn_sched_barrier(0);
  for (int b = 0;;) {
#pragma unroll 1
    for (int u = 0; u < UB && b + u < ft.nb; ++u) {
      const int band = __builtin_amdgcn_readlane(ft.band, b + u);
      const int sl = __builtin_amdgcn_readlane(ft.sl, b + u);
      const int ns = band >> 8, ol = band & 255;
      for (int o = 0; o < ol; ++o) xv[0] = shift_bin(n, xv[0]);
#pragma unroll 1
      for (int s0 = 0; s0 < ns; s0 += 4) {
        d2 mc[4], me[TWO ? 4 : 1];
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2) {
          const int s = sl + (s0 + s2 < ns ? s0 + s2 : ns - 1);
          mc[s2] = lds2(L.val, s, n.bin);
          if (TWO) me[TWO ? s2 : 0] = lds2(L.val, L.slots + s, n.bin);
        }
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2) {
          if (s0 + s2 < ns) {
            accB += mc[s2] * xv[0];
            if (TWO) accE += me[TWO ? s2 : 0] * xv[0];
            xv[0] = shift_bin(n, xv[0]);
          }
        }
      }
#pragma unroll
      for (int v = 0; v + 1 < UB; ++v) xv[v] = xv[v + 1];  // the next block's panel
    }
    b += UB;
    if (b >= ft.nb) break;
#pragma unroll
    for (int u = 0; u < UB; ++u)
      if (b + u < ft.nb)
        xv[u] = pload<SC1>(y, n.off, __builtin_amdgcn_readlane(ft.mo, b + u) * T.pb + cb);
  }
  if (TWO) accB += op.escale[k0 + n.half < kend ? k0 + n.half : kend - 1] * accE;
  acc[0] = acc[0] + accB;
  team_epilogue<1, TWO, REC>(op, st, T, L, si, stage, f0, ft.rc, ft.da, ft.slot, k0, kend, n, acc,
                             xo, fo, src);
}

// Per-lane descriptor of a dense-row wave: entry lane = one mother.
struct DenseDesc {
  // LDS slot and (first diagonal | diagonals << 8) per dense row; the second row
  // has single diagonals only
  int mo, s0, b0, s1, b1;
  double cw;  // Bethe-Heitler weight of the mother (EM sector)
};

// Partial sums of the dense rows over this wave's mothers (entries 0 .. ne-1 of
// its descriptor lanes) for the KP pairs of right-hand sides from k0.  The band row
// keeps one accumulator per diagonal, aligned with the mother's bins (its values
// are stored shifted by their diagonal, load_window): z_o[j] += v_o[j - o] x[j], and
// y[i] = sum_o z_o[i + o] once per stage -- 18 products per mother and pair
// instead of 18 and 7 shifts of 4 instructions.
// EM: also the Bethe-Heitler sum over the mothers, weight dd.cw each.
template <int KP, bool TWO, bool EM>
__device__ __forceinline__ void dense_partial(COp& op, __amdgpu_buffer_rsrc_t y, int pb,
                                              const TeamLds& L, const DenseDesc& dd, int ne, int k0,
                                              int kend, const Lane& n, d2 (&acc)[TSUMS][KP]) {
  constexpr int U = 2;
  d2 z[8][KP], w[KP], em[KP];
  double sc[KP];
#pragma unroll
  for (int p = 0; p < KP; ++p) {
#pragma unroll
    for (int o = 0; o < 8; ++o) z[o][p] = d2{0.0, 0.0};
    w[p] = em[p] = d2{0.0, 0.0};
    const int k = k0 + 2 * p + n.half;
    sc[p] = TWO ? op.escale[k < kend ? k : kend - 1] : 0.0;
  }
  const int cb = k0 * (WAVE * 8);
  for (int e = 0; e < ne; e += U) {
    d2 xv[U][KP];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int po = __builtin_amdgcn_readlane(dd.mo, (e + u) & 63) * pb + cb;
      const int vo = e + u < ne ? n.off : 0x7ffffff0;  // past the end: zeros
#pragma unroll
      for (int p = 0; p < KP; ++p) xv[u][p] = pload<SC1>(y, vo, po + p * (2 * WAVE * 8));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (e + u >= ne) break;
      if (EM) {
        const double cw = readlane_f64(dd.cw, e + u);
#pragma unroll
        for (int p = 0; p < KP; ++p) em[p] += cw * xv[u][p];
      }
      const int s0 = __builtin_amdgcn_readlane(dd.s0, e + u);
      const int b0 = __builtin_amdgcn_readlane(dd.b0, e + u);
      const int s1 = __builtin_amdgcn_readlane(dd.s1, e + u);
      const int b1 = __builtin_amdgcn_readlane(dd.b1, e + u);
      const int ns = b0 >> 8, ol = b0 & 255;
      // the diagonals in order; a row with fewer or later ones skips the others
#pragma unroll
      for (int o = 0; o < 8; ++o) {
        if (o >= ol && o < ol + ns) {
          const d2 mc = lds2(L.val, s0 + o - ol, n.bin);
          const d2 me = TWO ? lds2(L.val, L.slots + s0 + o - ol, n.bin) : d2{0.0, 0.0};
#pragma unroll
          for (int p = 0; p < KP; ++p) z[o][p] += (TWO ? mc + sc[p] * me : mc) * xv[u][p];
        }
      }
      if (b1 >> 8) {
        const d2 mc = lds2(L.val, s1, n.bin);
        const d2 me = TWO ? lds2(L.val, L.slots + s1, n.bin) : d2{0.0, 0.0};
#pragma unroll
        for (int p = 0; p < KP; ++p) w[p] += (TWO ? mc + sc[p] * me : mc) * xv[u][p];
      }
    }
  }
  // y = z_0 + shift(z_1 + shift(z_2 + ...)): seven shifts
#pragma unroll
  for (int p = 0; p < KP; ++p) {
    d2 t = z[7][p];
#pragma unroll
    for (int o = 6; o >= 0; --o) t = z[o][p] + shift_bin(n, t);
    acc[0][p] = t;
    acc[1][p] = w[p];
    acc[2][p] = em[p];
  }
}

// Arrive at and wait for a team barrier.  Stores of every wave have reached the
// coherence point before the arrival (vmcnt(0) of sc1 stores).  Returns false
// when the march is aborted.
__device__ __forceinline__ bool wait_count(const uint32_t* c, uint32_t target, uint32_t* abort_w,
                                           int limit) {
  int spins = 0;
  while (__hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
    if (++spins >= limit ||
        ((spins & 1023) == 0 &&
         __hip_atomic_load(abort_w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
      __hip_atomic_store(abort_w, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
  }
  return true;
}
__device__ __forceinline__ bool team_barrier(uint32_t* sub, uint32_t nsubwg, uint32_t* root,
                                             uint32_t nsub, uint32_t epoch, uint32_t* abort_w,
                                             int limit, int* bad) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (nsubwg * nsub == 1) return true;
  if (threadIdx.x == 0) {
    bool ok;
    if (nsub > 1) {
      const uint32_t old =
          __hip_atomic_fetch_add(sub, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (old + 1 == epoch * nsubwg)
        __hip_atomic_fetch_add(root, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ok = wait_count(root, epoch * nsub, abort_w, limit);
    } else {
      __hip_atomic_fetch_add(sub, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ok = wait_count(sub, epoch * nsubwg, abort_w, limit);
    }
    if (!ok) *bad = 1;
  }
  __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  return *bad == 0;
}
// (One arrival word per workgroup, polled with one vector load, measured the same at
// K = 1 and slower with more traffic: the pollers and writers share the lines.)

__global__ void team_reset(uint32_t* sync) {
  for (int i = threadIdx.x; i < SY_WORDS; i += blockDim.x) sync[i] = 0;
}

// Where a workgroup stands in its team, and the team's sync words.
struct TeamPos {
  int rank, c0, cend;  // right-hand sides [c0, cend) of the team
  int wv;
  Lane n;
  uint32_t *sub, *root, *abort_w;
  uint32_t nsub, nsubwg;
  int limit;  // polls of a wait
  int* bad;
};

__device__ __forceinline__ bool next_phase(const TeamPos& P, uint32_t& epoch) {
  return team_barrier(P.sub, P.nsubwg, P.root, P.nsub, ++epoch, P.abort_w, P.limit,
                      P.bad);
}

template <bool REC>
__device__ __forceinline__ StepIn step_in(CSch& sch, CSt& st, int step) {
  StepIn si;
  si.step = step;
  si.dl = cload(sch.dldz + step);
  si.h = cload(sch.h + step);
  si.hadia = cload(sch.hadia + step);
  si.finj = cload(sch.finj + step);
  si.ridx = REC && step - st.rec_first < st.rec_count ? step - st.rec_first : -1;
  return si;
}

// This workgroup's coupling values and the pair rate of window w into LDS (the
// caller puts barriers around it).
template <bool TWO>
__device__ __forceinline__ void load_window(COp& op, CTm& tm,
                                            const TeamLds& L, const TeamPos& P, int w) {
  const double* mv = op.mvals + (int64_t)w * op.mvals_stride;
  const double* me = TWO ? op.mvals_e + (int64_t)w * op.mvals_stride : nullptr;
  const int* vo = tm.lds_voff + 2 * cload(tm.lds_ptr + P.rank);
  const int lane = P.n.id;
#pragma unroll 4
  for (int s = P.wv; s < L.slots; s += TWAVES) {
    // value offset of the slot and by how many bins it is stored shifted
    const int v = cload(vo + 2 * s) + lane, sh = cload(vo + 2 * s + 1);
    const int at = lane + sh < WAVE ? lane + sh : lane + sh - WAVE;  // the wrapped bins: zeros
    L.val[s * WAVE + at] = lane + sh < WAVE ? mv[v] : 0.0;
    if (TWO) L.val[(L.slots + s) * WAVE + at] = lane + sh < WAVE ? me[v] : 0.0;
  }
  if (P.wv == 0) {
    L.rp[lane] = op.rpair[(int64_t)w * WAVE + lane];
    if (TWO) L.rp[WAVE + lane] = op.rpair_e[(int64_t)w * WAVE + lane];
  }
}

__device__ __forceinline__ RowTask row_task(COp& op, CTm& tm, int t,
                                            int lane, int pb) {
  const int* tk = tm.rows + 10 * t;
  RowTask r;
  r.a = cload(tk);
  r.b = cload(tk + 1);
  r.n2 = cload(tk + 2);
  r.na = cload(tk + 3);
  r.nb = cload(tk + 4);
  r.diag_a = cload(tk + 5);
  r.diag_b = cload(tk + 6);
  const int pa = cload(tk + 7), pq = cload(tk + 8), first = cload(tk + 9);
  r.part_a = pa < 0 ? -1 : pa * pb;
  r.part_b = pq < 0 ? -1 : pq * pb;
  r.ca = row_const(op, r.a);
  r.cb = row_const(op, r.b < 0 ? r.a : r.b);
  r.mo = r.sl = 0;
  if (lane < r.n2 + r.na + r.nb) {
    const int* q = tm.mothers + 2 * (first + lane);
    r.mo = q[0];
    r.sl = q[1];
  }
  return r;
}

// The state descriptors of this phase.
__device__ __forceinline__ TeamState team_state(CArgs* a) {
  TeamState T;
  T.pb = a->op.K * WAVE * 8;
  T.x = tile_rsrc(a->st.x, a->op.nspec * T.pb);
  T.a = tile_rsrc(a->st.a, a->op.nspec * T.pb);
  T.f = tile_rsrc(a->st.fphi, a->op.nspec * T.pb);
  T.phalf = a->tm.nparts * T.pb;
  T.part = tile_rsrc(a->tm.dpart, 2 * T.phalf);
  return T;
}

// March of a workgroup of rows: wave wv's tasks.  R = 2: row pairs, KP pairs of
// right-hand sides a pass, two waves per task (each every second pass).
template <int R, int KP, bool TWO, bool REC, bool SPLIT, bool EM>
__device__ __forceinline__ void march_rows(CArgs* A, const TeamLds& L, const TeamPos& P) {
  const int k_begin = A->k_begin, k_end = A->k_end;
  const int* wt = A->tm.wave_ptr + P.rank * TWAVES + P.wv;
  const int t0 = cload(wt), t1 = cload(wt + 1);
  RowTask first{};  // most waves have one task: it stays in registers
  if (t0 < t1) first = row_task(A->op, A->tm, t0, P.n.id, A->op.K * WAVE * 8);
  uint32_t epoch = 0;
  int wcur = -1;
  const int nc = P.cend - P.c0;
  coef_stage(L, k_begin, coef_ahead(A->op, A->sch, k_begin, P.c0, nc));
  __syncthreads();
#pragma unroll 1
  for (int p = 2 * k_begin; p < 2 * k_end; ++p) {
    CArgs* a = reread(A);
    const int s2 = p & 1, step = p >> 1;
    const int nx = step + 1 < k_end ? step + 1 : step;
    const bool ahead = s2 && P.wv * WAVE < L.coefs;
    const double cn = ahead ? coef_ahead(a->op, a->sch, nx, P.c0, nc) : 0.0;
    if (s2 == 0) {
      const int w = cload(a->sch.win + step);
      if (w != wcur) {
        __syncthreads();
        load_window<TWO>(a->op, a->tm, L, P, w);
        wcur = w;
        __syncthreads();
      }
    }
    const StepIn si = step_in<REC>(a->sch, a->st, step);
    const TeamState T = team_state(a);
#pragma unroll 1
    for (int t = t0; t < t1; ++t) {
      RowTask rt = first;
      if (t != t0) rt = row_task(a->op, a->tm, t, P.n.id, T.pb);
      if constexpr (R == 1) {
        team_row1<TWO, REC, SPLIT>(a->op, a->sch, a->st, T, L, si, s2, rt, P.c0, P.cend, P.n);
      } else {
        RowFactors fa{}, fb{};
        if (!TWO) {
          if (rt.part_a < 0)
            fa = row_factors<false>(a->op, L, si, s2, rt.ca.pscale, rt.diag_a, P.c0, P.n);
          if (rt.b >= 0 && rt.part_b < 0)
            fb = row_factors<false>(a->op, L, si, s2, rt.cb.pscale, rt.diag_b, P.c0, P.n);
        }
#pragma unroll 1
        for (int k0 = P.c0 + 2 * KP * (P.wv & 1); k0 < P.cend; k0 += 4 * KP)
          team_rows<KP, TWO, REC>(a->op, a->sch, a->st, T, L, si, s2, rt, fa, fb, P.c0, k0, P.cend,
                                  P.n);
      }
    }
    if (s2 && nx != step) coef_stage(L, nx, cn);  // complete behind the phase's barriers
    if (!next_phase(P, epoch)) return;
  }
  if (EM) next_phase(P, epoch);
}

// One stage's partial sums of a dense-row workgroup, KP pairs of right-hand
// sides per wave: mother group dg, column group dc.  Sum r of rank g is partial
// nsum g + r.
template <int KP, bool TWO, bool EM>
__device__ __forceinline__ void dense_stage_partials(COp& op, CTm& tm, const TeamState& T,
                                                     const TeamLds& L, const TeamPos& P,
                                                     __amdgpu_buffer_rsrc_t y, int pbase,
                                                     const DenseDesc& dd, int ne, int dg, int dc) {
  constexpr int NS = EM ? TSUMS : TDENSE;
  const int dG = tm.dgroups, dC = TWAVES / dG;
  const int po = pbase + P.rank * NS * T.pb;
  d2* const red = reinterpret_cast<d2*>(L.red);
  for (int k0 = P.c0 + dc * 2 * KP; k0 < P.cend; k0 += dC * 2 * KP) {
    d2 acc[TSUMS][KP];
    dense_partial<KP, TWO, EM>(op, y, T.pb, L, dd, ne, k0, P.cend, P.n, acc);
#pragma unroll
    for (int r = 0; r < NS; ++r)
#pragma unroll
      for (int p = 0; p < KP; ++p) {
        if (KP == 1 && dG > 1)
          red[(P.wv * NS + r) * WAVE + P.n.id] = acc[r][p];
        else if (k0 + 2 * p + P.n.half < P.cend)
          pstore<SC1>(acc[r][p], T.part, P.n.off, po + r * T.pb + (k0 + 2 * p) * (WAVE * 8));
      }
  }
  if (KP == 1 && dG > 1) {  // one column pass (2 dC covers the columns): add the mother groups in order
    __syncthreads();
    const int k0 = P.c0 + dc * 2;
    for (int r = dg; r < NS; r += dG) {
      if (k0 >= P.cend) break;
      d2 s = {0.0, 0.0};
      for (int g = 0; g < dG; ++g) s += red[((g * dC + dc) * NS + r) * WAVE + P.n.id];
      if (k0 + P.n.half < P.cend)
        pstore<SC1>(s, T.part, P.n.off, po + r * T.pb + k0 * (WAVE * 8));
    }
  }
}

// March of a dense-row workgroup: partial sums over its mothers.
template <int KD, bool TWO, bool EM>
__device__ __forceinline__ void march_dense(CArgs* A, const TeamLds& L, const TeamPos& P) {
  const int k_begin = A->k_begin, k_end = A->k_end;
  const int dG = A->tm.dgroups, dC = TWAVES / dG;
  const int dg = P.wv / dC, dc = P.wv % dC;
  const int* ep = A->tm.dense_ptr + P.rank * dG + dg;
  const int e0 = cload(ep), ne = cload(ep + 1) - e0;
  DenseDesc dd{0, 0, 0, 0, 0, 0.0};
  if (P.n.id < ne) {
    const int* q = A->tm.dense_ent + 5 * (e0 + P.n.id);
    dd = DenseDesc{q[0], q[1], q[2], q[3], q[4], EM ? A->tm.cbh[q[0]] : 0.0};
  }
  uint32_t epoch = 0;
  int wcur = -1;
  // with an EM sector one phase more: the weights of the last step's state
#pragma unroll 1
  for (int p = 2 * k_begin; p < 2 * k_end + (EM ? 1 : 0); ++p) {
    CArgs* a = reread(A);
    const int s2 = p & 1;
    if (s2 == 0 && p < 2 * k_end) {
      const int w = cload(a->sch.win + (p >> 1));
      if (w != wcur) {
        __syncthreads();
        load_window<TWO>(a->op, a->tm, L, P, w);
        wcur = w;
        __syncthreads();
      }
    }
    const TeamState T = team_state(a);
    dense_stage_partials<KD, TWO, EM>(a->op, a->tm, T, L, P, s2 ? T.a : T.x, s2 ? T.phalf : 0, dd, ne,
                                  dg, dc);
    if (!next_phase(P, epoch)) return;
  }
}

// sum_s cbh[s] x[s] for the pair of right-hand sides from k0 into slot step of the
// march's weights ([step - em_first][K][64]).
__device__ __forceinline__ void em_weights(CTm& tm, const TeamState& T, int step, int K, int k0,
                                           int kend, const Lane& n) {
  const int cb = k0 * (WAVE * 8);
  d2 s = {0.0, 0.0};
#pragma unroll 4
  for (int g = 0; g < tm.ndwg; ++g)
    s += pload<SC1>(T.part, n.off, (g * TSUMS + TDENSE) * T.pb + cb);
  for (int f = 0; f < tm.nfin; ++f) {
    const int da = cload(tm.fin + 8 * f);
    s += cload(tm.cbh + da) * pload<SC1>(T.x, n.off, da * T.pb + cb);
  }
  const int k = k0 + n.half;
  if (k < kend)
    *reinterpret_cast<d2*>(tm.em_w + ((int64_t)(step - tm.em_first) * K + k) * WAVE + n.bin) = s;
}

// March of a finishing workgroup: the tail rows, one stage behind the others.
template <bool TWO, bool REC, bool EM>
__device__ __forceinline__ void march_finish(CArgs* A, const TeamLds& L, const TeamPos& P) {
  constexpr int NF = TWO ? 2 : 1;
  const int k_begin = A->k_begin, k_end = A->k_end;
  const int groups = (P.cend - P.c0 + 1) / 2;
  const int items = A->tm.nfin * groups;
  const int it0 = (P.rank - A->tm.ndwg) * TWAVES + P.wv;
  const int stride = A->tm.nfwg * TWAVES;
  uint32_t epoch = 0;
  int wcur = -1, buf = 0;
  auto set = [&](int b) {  // LDS of value set b
    TeamLds Q = L;
    Q.val = L.val + b * NF * L.slots * WAVE;
    Q.rp = L.rp + b * NF * WAVE;
    return Q;
  };
  FinTask first{};
  if (it0 < items) first = fin_task(A->op, A->tm, it0 / groups, P.n.id);
  // phase p finishes stage p - 1: stage 2 of the step before, or stage 1 of its
  // own; sbuf: the value set of that stage
  int sbuf = 0;
  const int nc = P.cend - P.c0;
  constexpr int X = EM ? 1 : 0;  // the EM weights of the last step take a phase more
#pragma unroll 1
  for (int p = 2 * k_begin; p <= 2 * k_end + X; ++p) {
    CArgs* a = reread(A);
    const int s2 = (p & 1) ^ 1;
    // the step that its next phase begins to finish
    const bool ahead = s2 && p < 2 * k_end && P.wv * WAVE < L.coefs;
    const double cn = ahead ? coef_ahead(a->op, a->sch, p >> 1, P.c0, nc) : 0.0;
    sbuf = buf;
    if (s2 && p < 2 * k_end) {
      const int w = cload(a->sch.win + (p >> 1));
      if (w != wcur) {
        // into the other set: the last one is still read for the step before; the
        // phase's workgroup barriers complete it
        buf ^= 1;
        load_window<TWO>(a->op, a->tm, set(buf), P, w);
        wcur = w;
      }
    }
    if (EM && !s2 && (p >> 1) > k_begin) {
      // Bethe-Heitler sums of the state after step (p >> 1) - 1, which this phase
      // has whole: the partials of the heavy mothers and the tail rows' x
      const TeamState T = team_state(a);
#pragma unroll 1
      for (int g = it0; g < groups; g += stride)
        em_weights(a->tm, T, (p >> 1) - 1, a->op.K, P.c0 + 2 * g, P.cend, P.n);
    }
    if (p > 2 * k_begin && p <= 2 * k_end) {
      const TeamLds Q = set(sbuf);
      const StepIn si = step_in<REC>(a->sch, a->st, (p - 1) >> 1);
      const TeamState T = team_state(a);
#pragma unroll 1
      for (int it = it0; it < items; it += stride) {
        const int f = it / groups;
        FinTask ft = first;
        if (it != it0) ft = fin_task(a->op, a->tm, f, P.n.id);
        team_finish<TWO, REC>(a->op, a->sch, a->st, T, Q, si, s2, ft, P.c0,
                              P.c0 + (it - f * groups) * 2, P.cend, P.n);
      }
    }
    if (s2 && p < 2 * k_end) coef_stage(L, p >> 1, cn);
    if (p < 2 * k_end + X && !next_phase(P, epoch)) return;
  }
}

template <int R, int KP, int KD, bool TWO, bool REC, bool SPLIT, bool EM>
__global__ void __launch_bounds__(TTHREADS) team_march(TeamArgs) {
  extern __shared__ __attribute__((aligned(16))) double lds[];  // 16-byte reads
  __shared__ int bad;
  CArgs* const A = reinterpret_cast<CArgs*>(
      reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr()));
  const int K = A->op.K, nteam = A->tm.nteam, size = A->tm.size;
  const int team = (int)blockIdx.x % nteam;
  TeamPos P;
  P.rank = (int)blockIdx.x / nteam;
  P.n = lane_of();
  P.wv = wave_id();
  const int per = K / nteam, rem = K % nteam;
  P.c0 = team * per + (team < rem ? team : rem);
  P.cend = P.c0 + per + (team < rem ? 1 : 0);
  if (P.c0 == P.cend) return;  // uniform over the team: none of its workgroups waits

  TeamLds L;
  L.cst = lds;
  L.rp = L.cst + TCONST * WAVE;
  L.red = L.rp + (TWO ? 4 : 2) * WAVE;
  L.coef = L.red + A->tm.red_slots * WAVE;
  L.coefs = A->tm.coef_slots * WAVE;
  L.val = L.coef + 2 * L.coefs;
  L.slots = cload(A->tm.lds_ptr + P.rank + 1) - cload(A->tm.lds_ptr + P.rank);
  for (int i = threadIdx.x; i < WAVE; i += TTHREADS) {
    for (int o = 0; o < 7; ++o)  // zero where the neighbour lies outside the grid (team_epilogue)
      L.cst[o * WAVE + i] = (A->op.flags & PRH_F_PARTIAL_DIFF) && (unsigned)(i + o - 3) < WAVE
                                ? A->op.dcoef[i * 7 + o]
                                : 0.0;
    L.cst[7 * WAVE + i] = A->op.egrid[i];
    L.cst[8 * WAVE + i] = A->op.ddiag[i];
  }
  if (threadIdx.x == 0) bad = 0;
  P.bad = &bad;

  P.nsub = size > 32 ? size / 32 : 1;
  P.nsubwg = (uint32_t)size / P.nsub;
  P.sub = A->tm.sync + SY_SUB + (team * 8 + P.rank % P.nsub) * 64;
  P.root = A->tm.sync + SY_ROOT + team * 64;
  P.abort_w = A->tm.sync + SY_ABORT;
  P.limit = A->tm.spin_limit > 0 ? A->tm.spin_limit : SPIN_LIMIT;
  __syncthreads();

  const int ndwg = A->tm.ndwg, nfwg = A->tm.nfwg;
  if (P.rank < ndwg)
    march_dense<KD, TWO, EM>(A, L, P);
  else if (P.rank < ndwg + nfwg)
    march_finish<TWO, REC, EM>(A, L, P);
  else
    march_rows<R, KP, TWO, REC, SPLIT, EM>(A, L, P);
}

// Behind a march: NaN for the state, the recorded stage vectors and the EM weights
// of an aborted one.
__device__ __forceinline__ void fill_nan(double* p, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    p[i] = __builtin_nan("");
}
__global__ void team_void(TeamArgs a) {
  if (a.tm.sync[SY_ABORT] == 0) return;
  const int64_t panel = (int64_t)a.op.K * WAVE, nk = a.op.nspec * panel;
  fill_nan(a.st.x, nk);
  if (a.st.rec_x) {
    fill_nan(a.st.rec_x, a.st.rec_count * nk);
    fill_nan(a.st.rec_a, a.st.rec_count * nk);
    fill_nan(a.st.rec_fx, a.st.rec_count * nk);
    fill_nan(a.st.rec_fa, a.st.rec_count * nk);
  }
  if (a.tm.em_w)
    fill_nan(a.tm.em_w + (a.k_begin - a.tm.em_first) * panel, (a.k_end - a.k_begin) * panel);
}

// ---------------------------------------------------------------------------
// Adjoint sweep of a range of steps (the transposed stages of prh_adjoint_step) as
// one cooperative launch: teams, LDS values and barriers as above.  A transposed
// row reads at most a dozen lighter species by diagonal blocks and the protons by
// one band left of the diagonal, so there are no dense rows: a wave takes one row
// and a share of the team's columns.  u and v cross workgroups (sc1); lam, lam_a,
// the records and the accumulators belong to the row's wave.
// Per (row, pair of columns) and stage the two fields' factors cost about 250 of
// 400 vector instructions (two exponentials per bin in stage 2); the launches and
// their gaps were 65 us a stage at K = 64.
struct AdjArgs {
  prh_operator op;
  prh_schedule sch;
  prh_adjoint adj;
  prh_team tm;
  int k_begin, k_end;
};
typedef CONST_SPACE AdjArgs CAdjArgs;
__device__ __forceinline__ CAdjArgs* reread(CAdjArgs* a) {
  asm volatile("" : "+s"(a));
  return a;
}

__device__ __forceinline__ double dphi1_of(double z, double e, double p1) {
  return (fabs(z) < 1e-2) ? 0.5 + z * (1.0 / 3.0 + z * (1.0 / 8.0 + z * (1.0 / 30.0)))
                          : (e - p1) / z;
}
__device__ __forceinline__ double dphi2_of(double z, double p1, double p2) {
  return (fabs(z) < 1e-2) ? 1.0 / 6.0 + z * (1.0 / 12.0 + z * (1.0 / 40.0 + z * (1.0 / 180.0)))
                          : (p1 - 2.0 * p2) / z;
}
// the panel moved up by one bin: bin i receives bin i - 1
__device__ __forceinline__ d2 shift_bin_up(const Lane& n, d2 v) { return d2{prev1(n, v.y), v.x}; }

// kappa, h d of a row and column at one bin, and their field parts
struct BinCoef {
  double kap, kapE, hd, dE;
};
template <bool TWO>
__device__ __forceinline__ BinCoef bin_coef(double kadia, double pscale, double rc, double re,
                                            double mdc, double mde, double ddiag, double s,
                                            double dl, double h, bool pdiff) {
  BinCoef b;
  b.kap = kadia + pscale * (TWO ? rc + s * re : rc);
  b.kapE = TWO ? pscale * re : 0.0;
  double dval = (TWO ? mdc + s * mde : mdc) * dl;
  if (pdiff) {
    double kxd = b.kap * ddiag;
    kxd = kxd * dl;
    dval = dval + kxd;
  }
  b.hd = dval * h;
  b.dE = TWO ? (mde + b.kapE * ddiag) * dl : 0.0;
  return b;
}

// A transposed row of a wave; lane e holds entry e: mother, LDS slot, and for a
// band its first diagonal (negative) and number of diagonals.
struct AdjRow {
  int r, nd, nb, slot, cg, ncg;
  double pscale;
  int sslot;
  int mo, sl, ol, ns;
};

template <bool TWO>
__device__ __forceinline__ void adjoint_row(CAdjArgs* a, const TeamLds& L, const TeamState& T,
                                            const AdjRow& ar, int s2, int step, int c0, int k0,
                                            int kend, const Lane& n) {
  constexpr int U = 6;
  const auto y = s2 ? T.a : T.x;  // v or u
  const int K = a->op.K;
  const int cb = k0 * (WAVE * 8);
  const int own = ar.r * T.pb + cb;
  const int k = k0 + n.half;
  const int kc = k < kend ? k : kend - 1;
  const int64_t oi = ((int64_t)ar.r * K + kc) * WAVE + n.bin;
  const bool pdiff = (a->op.flags & PRH_F_PARTIAL_DIFF) != 0;
  d2 acc = {0.0, 0.0}, accE = acc;
  const d2 yo = pload<SC1>(y, n.off, own);
  const d2 lp = *reinterpret_cast<const d2*>((s2 ? a->adj.lam_a : a->adj.lam) + oi);
  // diagonal blocks
#pragma unroll 1
  for (int e = 0; e < ar.nd; e += U) {
    d2 xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int po = __builtin_amdgcn_readlane(ar.mo, (e + u) & 63) * T.pb + cb;
      xv[u] = pload<SC1>(y, e + u < ar.nd ? n.off : 0x7ffffff0, po);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (e + u < ar.nd) {
        const int sl = __builtin_amdgcn_readlane(ar.sl, e + u);
        acc += lds2(L.val, sl, n.bin) * xv[u];
        if (TWO) accE += lds2(L.val, L.slots + sl, n.bin) * xv[u];
      }
    }
  }
  // bands: every diagonal at or left of the main one, walked from the last
#pragma unroll 1
  for (int e = ar.nd; e < ar.nd + ar.nb; ++e) {
    const int sl = __builtin_amdgcn_readlane(ar.sl, e);
    const int ol = __builtin_amdgcn_readlane(ar.ol, e), ns = __builtin_amdgcn_readlane(ar.ns, e);
    d2 x = pload<SC1>(y, n.off, __builtin_amdgcn_readlane(ar.mo, e) * T.pb + cb);
    for (int o = ol + ns - 1; o < 0; ++o) x = shift_bin_up(n, x);
#pragma unroll 1
    for (int q0 = ns - 1; q0 >= 0; q0 -= 4) {
      d2 mc[4], me[TWO ? 4 : 1];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int sq = sl + (q0 - q >= 0 ? q0 - q : 0);
        mc[q] = lds2(L.val, sq, n.bin);
        if (TWO) me[TWO ? q : 0] = lds2(L.val, L.slots + sq, n.bin);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q0 - q >= 0) {
          acc += mc[q] * x;
          if (TWO) accE += me[TWO ? q : 0] * x;
          x = shift_bin_up(n, x);
        }
      }
    }
  }
  const double s = TWO ? a->op.escale[kc] : 0.0;
  const double dl = cload(a->sch.dldz + step), hh = cload(a->sch.h + step);
  const double hadia = cload(a->sch.hadia + step);
  // transposed FD stencil D^T y, neighbours -3 .. 3 in order
  d2 q = {0.0, 0.0};
  if (pdiff) {
    const double m1 = prev1(n, yo.y), m2 = prev1(n, yo.x), m3 = prev1(n, m1);
    const double p2 = next1(n, yo.x), p3 = next1(n, yo.y), p4 = next1(n, p2);
    q += lds2(L.cst, 0, n.bin) * d2{m3, m2};
    q += lds2(L.cst, 1, n.bin) * d2{m2, m1};
    q += lds2(L.cst, 2, n.bin) * d2{m1, yo.x};
    q += lds2(L.cst, 4, n.bin) * d2{yo.y, p2};
    q += lds2(L.cst, 5, n.bin) * d2{p2, p3};
    q += lds2(L.cst, 6, n.bin) * d2{p3, p4};
  }
  const d2 mty = TWO ? acc + s * accE : acc;
  const bool want_s = TWO && a->adj.gdot != nullptr;
  const int64_t nk = (int64_t)a->op.nspec * K * WAVE;
  const int64_t ri = (step - a->adj.rec_first) * nk + oi;
  d2 xx = {0.0, 0.0}, xa = xx, fx = xx, fa = xx, gd = xx;
  if (want_s) {
    xx = *reinterpret_cast<const d2*>(a->adj.rec_x + ri);
    gd = *reinterpret_cast<const d2*>(a->adj.gdot + oi);
    if (!s2) {
      xa = *reinterpret_cast<const d2*>(a->adj.rec_a + ri);
      fx = *reinterpret_cast<const d2*>(a->adj.rec_fx + ri);
      fa = *reinterpret_cast<const d2*>(a->adj.rec_fa + ri);
    }
  }
  // the step before, for u (its window may be another one: from memory)
  double dlp = 0.0, hp = 0.0, hadp = 0.0;
  d2 pmc = {0.0, 0.0}, pme = pmc, prc = pmc, pre = pmc;
  if (s2 && step > 0) {
    const int sp = step - 1;
    const int64_t wp = cload(a->sch.win + sp);
    dlp = cload(a->sch.dldz + sp);
    hp = cload(a->sch.h + sp);
    hadp = cload(a->sch.hadia + sp);
    const int64_t dg = wp * a->op.mvals_stride + a->op.diag_off + (int64_t)ar.r * WAVE + n.bin;
    pmc = *reinterpret_cast<const d2*>(a->op.mvals + dg);
    prc = *reinterpret_cast<const d2*>(a->op.rpair + wp * WAVE + n.bin);
    if (TWO) {
      pme = *reinterpret_cast<const d2*>(a->op.mvals_e + dg);
      pre = *reinterpret_cast<const d2*>(a->op.rpair_e + wp * WAVE + n.bin);
    }
  }
  const d2 eg = lds2(L.cst, 7, n.bin), dd = lds2(L.cst, 8, n.bin);
  const d2 rc = lds2(L.rp, 0, n.bin), mdc = lds2(L.val, ar.slot, n.bin);
  const d2 re = TWO ? lds2(L.rp, 1, n.bin) : d2{0.0, 0.0};
  const d2 mde = TWO ? lds2(L.val, L.slots + ar.slot, n.bin) : d2{0.0, 0.0};
  d2 out0, out1, wv, gs;  // new lam_a and v (stage 1), lam and u (stage 2)
#pragma unroll 1
  for (int b = 0; b < 2; ++b) {  // one bin after the other: half the code
    auto at = [&](const d2& v) { return b ? v.y : v.x; };
    const BinCoef c = bin_coef<TWO>(hadia * at(eg), ar.pscale, at(rc), at(re), at(mdc), at(mde),
                                    at(dd), s, dl, hh, pdiff);
    const double e = exp(c.hd);
    const double t = (at(mty) + c.kap * at(q)) * dl;
    double o0, o1, g = 0.0, ww = 0.0;
    if (!s2) {
      const double p1 = phi1_of(c.hd, e), p2 = phi2_of(c.hd, e);
      o0 = at(lp) + t;
      ww = hh * p1 * o0;
      o1 = ww - at(yo);
      if (want_s) {
        g = dl * (at(accE) + c.kapE * at(q)) * at(xa);
        const double dJdd = o0 * (hh * e * at(xx) + hh * hh * dphi1_of(c.hd, e, p1) * at(fx)) +
                            at(lp) * (hh * hh * dphi2_of(c.hd, p1, p2) * (at(fa) - at(fx)));
        g += dJdd * c.dE;
      }
    } else {
      o0 = e * at(lp) + t;
      if (want_s) g = dl * (at(accE) + c.kapE * at(q)) * at(xx);
      const BinCoef cp = bin_coef<TWO>(hadp * at(eg), ar.pscale, at(prc), at(pre), at(pmc), at(pme),
                                       at(dd), s, dlp, hp, pdiff);
      o1 = hp * phi2_of(cp.hd, exp(cp.hd)) * o0;
    }
    if (b) {
      out0.y = o0;
      out1.y = o1;
      gs.y = g;
      wv.y = ww;
    } else {
      out0.x = o0;
      out1.x = o1;
      gs.x = g;
      wv.x = ww;
    }
  }
  if (k >= kend) return;  // the odd last right-hand side's idle half
  *reinterpret_cast<d2*>((s2 ? a->adj.lam : a->adj.lam_a) + oi) = out0;
  if (!s2)
    pstore<SC1>(out1, T.a, n.off, own);
  else if (step > 0)
    pstore<SC1>(out1, T.x, n.off, own);
  if (want_s) *reinterpret_cast<d2*>(a->adj.gdot + oi) = gd + gs;
  if (!s2 && ar.sslot >= 0) {
    const double f = cload(a->sch.finj + step), lz = cload(a->adj.lnz1 + step);
    const int J = a->op.nsrc, nc = kend - c0;
    for (int j = 0; j < J; ++j) {
      const double c = L.coef[(step & 1) * L.coefs + j * nc + k - c0];
      const int64_t gi = (((int64_t)ar.sslot * J + j) * K + k) * WAVE + n.bin;
      d2* g0 = reinterpret_cast<d2*>(a->adj.gsrc0 + gi);
      d2* g1 = reinterpret_cast<d2*>(a->adj.gsrc1 + gi);
      *g0 += f * c * wv;
      *g1 += f * c * lz * wv;
    }
  }
}

template <bool TWO>
__global__ void __launch_bounds__(TTHREADS) adjoint_march(AdjArgs) {
  extern __shared__ __attribute__((aligned(16))) double lds[];
  __shared__ int bad;
  CAdjArgs* const A = reinterpret_cast<CAdjArgs*>(
      reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr()));
  const int K = A->op.K, nteam = A->tm.nteam, size = A->tm.size;
  const int team = (int)blockIdx.x % nteam;
  TeamPos P;
  P.rank = (int)blockIdx.x / nteam;
  P.n = lane_of();
  P.wv = wave_id();
  const int per = K / nteam, rem = K % nteam;
  P.c0 = team * per + (team < rem ? team : rem);
  P.cend = P.c0 + per + (team < rem ? 1 : 0);
  if (P.c0 == P.cend) return;
  TeamLds L;
  L.cst = lds;
  L.rp = L.cst + TCONST * WAVE;
  L.red = nullptr;
  L.coef = L.rp + (TWO ? 2 : 1) * WAVE;
  L.coefs = A->tm.coef_slots * WAVE;
  L.val = L.coef + 2 * L.coefs;
  L.slots = cload(A->tm.lds_ptr + P.rank + 1) - cload(A->tm.lds_ptr + P.rank);
  for (int i = threadIdx.x; i < WAVE; i += TTHREADS) {
    for (int o = 0; o < 7; ++o)  // zero where the neighbour lies outside the grid (team_epilogue)
      L.cst[o * WAVE + i] = (A->op.flags & PRH_F_PARTIAL_DIFF) && (unsigned)(i + o - 3) < WAVE
                                ? A->op.dcoef[i * 7 + o]
                                : 0.0;
    L.cst[7 * WAVE + i] = A->op.egrid[i];
    L.cst[8 * WAVE + i] = A->op.ddiag[i];
  }
  if (threadIdx.x == 0) bad = 0;
  P.bad = &bad;
  P.nsub = size > 32 ? size / 32 : 1;
  P.nsubwg = (uint32_t)size / P.nsub;
  P.sub = A->tm.sync + SY_SUB + (team * 8 + P.rank % P.nsub) * 64;
  P.root = A->tm.sync + SY_ROOT + team * 64;
  P.abort_w = A->tm.sync + SY_ABORT;
  P.limit = A->tm.spin_limit > 0 ? A->tm.spin_limit : SPIN_LIMIT;
  const int k_begin = A->k_begin, k_end = A->k_end;
  const int nc = P.cend - P.c0;
  const bool src = A->adj.gsrc0 != nullptr && (A->op.flags & PRH_F_INJECTION) != 0;
  if (src) coef_stage(L, k_end - 1, coef_ahead(A->op, A->sch, k_end - 1, P.c0, nc));
  __syncthreads();
  const int* wt = A->tm.wave_ptr + P.rank * TWAVES + P.wv;
  const int t0 = cload(wt), t1 = cload(wt + 1);
  uint32_t epoch = 0;
  int wcur = -1;
#pragma unroll 1
  for (int p = 2 * (k_end - k_begin) - 1; p >= 0; --p) {
    CAdjArgs* a = reread(A);
    const int s2 = (p & 1) ^ 1;  // stage 1 of a step, then stage 2
    const int step = k_begin + (p >> 1);
    const bool ahead = src && s2 && step > k_begin && P.wv * WAVE < L.coefs;
    const double cn = ahead ? coef_ahead(a->op, a->sch, step - 1, P.c0, nc) : 0.0;
    if (!s2) {
      const int w = cload(a->sch.win + step);
      if (w != wcur) {
        __syncthreads();
        load_window<TWO>(a->op, a->tm, L, P, w);
        wcur = w;
        __syncthreads();
      }
    }
    TeamState T;
    T.pb = K * WAVE * 8;
    T.x = tile_rsrc(a->adj.u, a->op.nspec * T.pb);
    T.a = tile_rsrc(a->adj.v, a->op.nspec * T.pb);
#pragma unroll 1
    for (int t = t0; t < t1; ++t) {
      const int* tk = a->tm.rows + 10 * t;
      AdjRow ar;
      ar.r = cload(tk);
      ar.nd = cload(tk + 1);
      ar.nb = cload(tk + 2);
      ar.slot = cload(tk + 3);
      ar.cg = cload(tk + 4);
      ar.ncg = cload(tk + 5);
      ar.pscale = cload(a->op.pscale + ar.r);
      ar.sslot = src ? cload(a->op.src_slot + ar.r) : -1;
      ar.mo = ar.sl = ar.ol = ar.ns = 0;
      if (P.n.id < ar.nd + ar.nb) {
        const int* q = a->tm.mothers + 4 * (cload(tk + 6) + P.n.id);
        ar.mo = q[0];
        ar.sl = q[1];
        ar.ol = q[2];
        ar.ns = q[3];
      }
#pragma unroll 1
      for (int k0 = P.c0 + 2 * ar.cg; k0 < P.cend; k0 += 2 * ar.ncg)
        adjoint_row<TWO>(a, L, T, ar, s2, step, P.c0, k0, P.cend, P.n);
    }
    if (ahead) coef_stage(L, step - 1, cn);
    if (!next_phase(P, epoch)) return;
  }
}

// Behind it: NaN for lam and the accumulators of an aborted sweep.
__global__ void adjoint_void(AdjArgs a) {
  if (a.tm.sync[SY_ABORT] == 0) return;
  const int64_t panel = (int64_t)a.op.K * WAVE, nk = a.op.nspec * panel;
  fill_nan(a.adj.lam, nk);
  if (a.adj.gdot) fill_nan(a.adj.gdot, nk);
  if (!a.adj.gsrc0 || !(a.op.flags & PRH_F_INJECTION)) return;
  for (int i = 0; i < a.op.nspec; ++i) {
    const int s = a.op.src_slot[i];
    if (s < 0) continue;
    fill_nan(a.adj.gsrc0 + s * (a.op.nsrc * panel), a.op.nsrc * panel);
    fill_nan(a.adj.gsrc1 + s * (a.op.nsrc * panel), a.op.nsrc * panel);
  }
}

// ---------------------------------------------------------------------------
// Photons of the co-evolved EM cascade over a range of steps.  The nuclei do not
// see the photons, so the march leaves only the Bethe-Heitler sums of each step
// and the photons follow here: per step out = [qstep | 2 T_e R_BH] [gam; bhw W]
// for every column by itself.  One workgroup carries 16 columns through all steps
// with the photons in LDS, one wave per 16 photon bins (FP64 MFMA); the
// registers of the step's matrix fragment are refilled with the next step's as
// each is used.  Bound by the FP64 MFMA rate of its CU, about 3 us a step
// (136 x 200 x 16), against 18.8 us a step for two launches over the whole
// batch at K = 512 and 8 us at K = 64.
constexpr int EMW_TILES = PRH_EM_MAX / 16;    // waves: 16-row tiles of the photon grid
constexpr int EMW_NQ = PRH_EM_MAX / 8;        // pairs of k-steps over the photons
constexpr int EMW_NW = WAVE / 8;              // and over the nucleon bins
constexpr int EMW_ROW = PRH_EM_MAX + WAVE + 2;  // LDS row of a column (padded)
typedef double d4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(EMW_TILES * WAVE)
    em_photon_march(prh_schedule sch, prh_em em, const double* __restrict__ wsum, int w_first, int K,
                    int k_begin, int k_end) {
  __shared__ __attribute__((aligned(16))) double y[2][16][EMW_ROW];
  const int de = em.d_em;
  const int kd = de + WAVE;
  const int nq = de / 8;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = wave_id();
  const int col = lane & 15, kq = lane >> 4;
  const int row = wv * 16 + col;                 // A operand: this lane's matrix row
  const int rowc = row < de ? row : de - 1;
  // columns' photons (rows past de stay zero) and the first step's weights
  const double* g0 = (k_begin & 1) ? em.gam2 : em.gam;
  for (int i = threadIdx.x; i < 16 * EMW_ROW; i += blockDim.x) {
    const int c = i / EMW_ROW, r = i % EMW_ROW;
    const int k = blockIdx.x * 16 + c;
    y[0][c][r] = (r < de && k < K) ? g0[(int64_t)r * K + k] : 0.0;
    y[1][c][r] = 0.0;
  }
  // weights of step t for this thread's (column, bin) pairs: 1024 over 576 threads
  constexpr int NT = EMW_TILES * WAVE;
  auto weight = [&](int t, int i) {
    const int c = i / WAVE, j = i % WAVE;
    const int k = blockIdx.x * 16 + c < K ? blockIdx.x * 16 + c : K - 1;
    return em.bhw[(int64_t)sch.win[t] * WAVE + j] *
           wsum[((int64_t)(t - w_first) * K + k) * WAVE + j];
  };
  auto fragment = [&](int t, int i) -> d2 {  // pair of k-steps i of step t
    if (i < nq)
      return *reinterpret_cast<const d2*>(em.qstep + ((int64_t)t * de + rowc) * de + 8 * i + 2 * kq);
    return *reinterpret_cast<const d2*>(em.tstack + ((int64_t)sch.win[t] * de + rowc) * kd + 8 * i +
                                        2 * kq);
  };
  d2 a[EMW_NQ + EMW_NW];
  const int np = nq + EMW_NW;
#pragma unroll
  for (int i = 0; i < EMW_NQ + EMW_NW; ++i)
    if (i < np) a[i] = fragment(k_begin, i);
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * WAVE; i += NT) y[0][i / WAVE][de + i % WAVE] = weight(k_begin, i);
  __syncthreads();
#pragma unroll 1
  for (int t = k_begin; t < k_end; ++t) {
    const int b = (t - k_begin) & 1;
    const int nx = t + 1 < k_end ? t + 1 : t;
    const double w0 = weight(nx, threadIdx.x);
    const double w1 = threadIdx.x + NT < 16 * WAVE ? weight(nx, threadIdx.x + NT) : 0.0;
    d4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = acc0;
#pragma unroll
    for (int i = 0; i < EMW_NQ + EMW_NW; ++i) {
      if (i < np) {
        const d2 v = *reinterpret_cast<const d2*>(&y[b][col][8 * i + 2 * kq]);
        acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, v.x, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, v.y, acc1, 0, 0, 0);
        a[i] = fragment(nx, i);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = wv * 16 + kq + 4 * v;
      if (r < de) y[b ^ 1][col][r] = acc0[v] + acc1[v];
    }
    y[b ^ 1][threadIdx.x / WAVE][de + threadIdx.x % WAVE] = w0;
    if (threadIdx.x + NT < 16 * WAVE)
      y[b ^ 1][(threadIdx.x + NT) / WAVE][de + threadIdx.x % WAVE] = w1;
    __syncthreads();
  }
  const int b = (k_end - k_begin) & 1;
  double* g1 = (k_end & 1) ? em.gam2 : em.gam;
  for (int i = threadIdx.x; i < 16 * de; i += blockDim.x) {
    const int r = i / 16, c = i % 16;
    const int k = blockIdx.x * 16 + c;
    if (k < K) g1[(int64_t)r * K + k] = y[b][c][r];
  }
}

// fn: the march; behind: the launch that voids an aborted one's results (same arguments)
int32_t launch_march(const void* fn, const void* behind, const prh_team& tm, size_t lds_rows,
                     void* kernel_args, hipStream_t s) {
  return prh_internal::launch_march(
      {reinterpret_cast<const void*>(&team_reset), fn, behind, (unsigned)(tm.nteam * tm.size),
       TTHREADS, 8 * WAVE * lds_rows, tm.sync, kernel_args},
      s);
}

// 0, or NOT_LAUNCHABLE when the stream is being captured (a cooperative launch cannot be)
int32_t refuse_capture(hipStream_t s) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (int32_t e = prh_internal::check(hipStreamIsCapturing(s, &cs), "team march: capture status"))
    return e;
  if (cs == hipStreamCaptureStatusNone) return 0;
  prh_internal::error("team march: a cooperative launch cannot be captured");
  return prh_internal::NOT_LAUNCHABLE;
}

template <int R, int KP, int KD, bool TWO, bool REC, bool SPLIT, bool EM>
int32_t launch_team_rec(const prh_operator& op, const prh_schedule& sch, const prh_state& st,
                        const prh_team& tm, int k_begin, int k_end, hipStream_t s) {
  TeamArgs ta{op, sch, st, tm, k_begin, k_end};
  return launch_march(reinterpret_cast<const void*>(&team_march<R, KP, KD, TWO, REC, SPLIT, EM>),
                      reinterpret_cast<const void*>(&team_void), tm,
                      (size_t)(TCONST + (TWO ? 4 : 2) + 2 * tm.coef_slots + tm.red_slots +
                               tm.lds_slots * (TWO ? 2 : 1)),
                      &ta, s);
}

template <int R, int KP, int KD, bool TWO, bool SPLIT>
int32_t launch_team(const prh_operator& op, const prh_schedule& sch, const prh_state& st,
                    const prh_team& tm, int k_begin, int k_end, hipStream_t s) {
  if constexpr (!TWO) {
    if (tm.em_w)
      return launch_team_rec<R, KP, KD, false, false, SPLIT, true>(op, sch, st, tm, k_begin, k_end,
                                                                  s);
  }
  return st.rec_x ? launch_team_rec<R, KP, KD, TWO, true, SPLIT, false>(op, sch, st, tm, k_begin,
                                                                       k_end, s)
                  : launch_team_rec<R, KP, KD, TWO, false, SPLIT, false>(op, sch, st, tm, k_begin,
                                                                        k_end, s);
}

}  // namespace

extern "C" int32_t prh_team_march(const prh_operator* op, const prh_schedule* sch,
                                  const prh_state* st, const prh_team* tm, int32_t k_begin,
                                  int32_t k_end, void* stream) {
  using prh_internal::error;
  if (!op || !sch || !st || !tm) return error("prh_team_march: null argument");
  if (op->d != WAVE) return error("prh_team_march: 64 energy bins only");
  if (op->K <= 0 || op->nspec <= 0) return error("prh_team_march: empty operator");
  // byte offsets of the state and of the partials are 32-bit
  if ((int64_t)op->nspec * op->K * WAVE * 8 > 0x7fffffff ||
      2 * (int64_t)tm->nparts * op->K * WAVE * 8 > 0x7fffffff)
    return error("prh_team_march: a state array exceeds 2 GiB");
  if ((op->mvals_e == nullptr) != (op->escale == nullptr) ||
      (op->mvals_e != nullptr && op->rpair_e == nullptr))
    return error("prh_team_march: mvals_e, rpair_e and escale go together");
  if (st->em) return error("prh_team_march: no EM sector");
  if (!st->x || !st->a || !st->fphi) return error("prh_team_march: null state");
  if (st->rec_x && (!st->rec_a || !st->rec_fx || !st->rec_fa))
    return error("prh_team_march: recording needs all four record arrays");
  if (k_begin < 0 || k_end > sch->nsteps || k_begin > k_end)
    return error("prh_team_march: step range outside the schedule");
  if (tm->nteam < 1 || tm->nteam > 8 || tm->size < 1 || tm->size > 256 ||
      (tm->size > 32 && tm->size % 32 != 0))
    return error("prh_team_march: 1 to 8 teams of up to 32 workgroups, or a multiple of 32");
  if (tm->ndwg < 0 || tm->nfwg < 0 || tm->nfin < 0 || tm->nparts < (tm->em_w ? TSUMS : TDENSE) * tm->ndwg ||
      tm->ndwg + tm->nfwg > tm->size || (tm->nfin > 0) != (tm->nfwg > 0))
    return error("prh_team_march: tail rows need finishing workgroups, all within the team");
  if (!tm->sync || !tm->rows || !tm->wave_ptr || !tm->mothers || !tm->lds_ptr || !tm->lds_voff)
    return error("prh_team_march: null table");
  if ((tm->ndwg > 0 && (!tm->dense_ptr || !tm->dense_ent)) ||
      (tm->nfin > 0 && (!tm->fin || !tm->fin_blk)) || (tm->nparts > 0 && !tm->dpart))
    return error("prh_team_march: tail rows need their tables and partials");
  if (tm->em_w && (!tm->cbh || tm->nfin < 1 || op->mvals_e || st->rec_x || k_begin < tm->em_first))
    return error("prh_team_march: EM weights need cbh, a tail row, one field and no recording");
  if (!(tm->kd == 1 || tm->kd == 2) || tm->dgroups < 1 || tm->dgroups > TWAVES ||
      TWAVES % tm->dgroups != 0)
    return error("prh_team_march: bad dense-row tiling");
  const int ncmax = (op->K + tm->nteam - 1) / tm->nteam;
  if (tm->ndwg > 0 && tm->dgroups > 1 &&
      (tm->dgroups < TDENSE || tm->kd != 1 || (TWAVES / tm->dgroups) * 2 < ncmax ||
       tm->red_slots < TWAVES * 2 * (tm->em_w ? TSUMS : TDENSE)))
    return error("prh_team_march: mother groups need one column pass and their LDS rows");
  if (op->nsrc * ncmax > TTHREADS || op->nsrc * ncmax > WAVE * tm->coef_slots)
    return error("prh_team_march: more source coefficients per team than staged");
  if (k_begin == k_end) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (int32_t e = refuse_capture(s)) return e;
  if (tm->pair_rows == 0 && ncmax > 2)
    return error("prh_team_march: single-row tasks take at most 2 right-hand sides per team");
  // one right-hand side per team: the halves of a wave share it
  const int key = tm->pair_rows == 0 ? ncmax : 10 * tm->kp + tm->kd;
#define TEAM(R, KP, KD, TWO, SPLIT) \
  return launch_team<R, KP, KD, TWO, SPLIT>(*op, *sch, *st, *tm, k_begin, k_end, s)
  if (op->mvals_e) {
    switch (key) {
      case 1: TEAM(1, 1, 1, true, true);
      case 2: TEAM(1, 1, 1, true, false);
      case 11: TEAM(2, 1, 1, true, false);
      case 21: TEAM(2, 2, 1, true, false);
      case 22: TEAM(2, 2, 2, true, false);
    }
  } else {
    switch (key) {
      case 1: TEAM(1, 1, 1, false, true);
      case 2: TEAM(1, 1, 1, false, false);
      case 11: TEAM(2, 1, 1, false, false);
      case 21: TEAM(2, 2, 1, false, false);
      case 22: TEAM(2, 2, 2, false, false);
    }
  }
#undef TEAM
  return error("prh_team_march: no kernel for this kp, kd");
}

extern "C" int32_t prh_em_photon_march(const prh_operator* op, const prh_schedule* sch,
                                       const prh_em* em, const double* wsum, int32_t w_first,
                                       int32_t k_begin, int32_t k_end, void* stream) {
  using prh_internal::error;
  if (!op || !sch || !em || !wsum) return error("prh_em_photon_march: null argument");
  if (op->d != WAVE || em->d_em < 8 || em->d_em > PRH_EM_MAX || em->d_em % 8 != 0)
    return error("prh_em_photon_march: 64 nucleon bins, EM bins a multiple of 8 up to 144");
  if (!em->gam || !em->gam2 || !em->bhw || !em->tstack || !em->qstep || op->K < 1)
    return error("prh_em_photon_march: EM sector with a null buffer");
  if (k_begin < 0 || k_end > sch->nsteps || k_begin > k_end || w_first < 0 || w_first > k_begin)
    return error("prh_em_photon_march: step range outside the schedule");
  if (k_begin == k_end) return 0;
  hipLaunchKernelGGL(em_photon_march, dim3((unsigned)((op->K + 15) / 16)), dim3(EMW_TILES * WAVE), 0,
                     (hipStream_t)stream, *sch, *em, wsum, (int)w_first, (int)op->K, (int)k_begin,
                     (int)k_end);
  return prh_internal::check(hipGetLastError(), "prh_em_photon_march launch");
}

extern "C" int32_t prh_team_adjoint(const prh_operator* op, const prh_schedule* sch,
                                    const prh_adjoint* adj, const prh_team* tm, int32_t k_begin,
                                    int32_t k_end, void* stream) {
  using prh_internal::error;
  if (!op || !sch || !adj || !tm) return error("prh_team_adjoint: null argument");
  if (op->d != WAVE) return error("prh_team_adjoint: 64 energy bins only");
  if (op->K <= 0 || op->nspec <= 0) return error("prh_team_adjoint: empty operator");
  if ((int64_t)op->nspec * op->K * WAVE * 8 > 0x7fffffff)
    return error("prh_team_adjoint: a state array exceeds 2 GiB");
  if ((op->mvals_e == nullptr) != (op->escale == nullptr) ||
      (op->mvals_e != nullptr && op->rpair_e == nullptr))
    return error("prh_team_adjoint: mvals_e, rpair_e and escale go together");
  if (!adj->lam || !adj->lam_a || !adj->u || !adj->v)
    return error("prh_team_adjoint: lam, lam_a, u and v are required");
  if (k_begin < 0 || k_end > sch->nsteps || k_begin > k_end)
    return error("prh_team_adjoint: step range outside the schedule");
  if (op->mvals_e && adj->gdot) {
    if (!adj->rec_x || !adj->rec_a || !adj->rec_fx || !adj->rec_fa)
      return error("prh_team_adjoint: the EBL-scale gradient needs the recorded forward steps");
    if (k_begin < adj->rec_first || k_end > adj->rec_first + adj->rec_count)
      return error("prh_team_adjoint: steps outside the recorded chunk");
  }
  if (adj->gsrc0 && (!adj->gsrc1 || !adj->lnz1))
    return error("prh_team_adjoint: source accumulators need gsrc1 and lnz1");
  if (tm->nteam < 1 || tm->nteam > 8 || tm->size < 1 || tm->size > 256 ||
      (tm->size > 32 && tm->size % 32 != 0))
    return error("prh_team_adjoint: 1 to 8 teams of up to 32 workgroups, or a multiple of 32");
  if (!tm->sync || !tm->rows || !tm->wave_ptr || !tm->mothers || !tm->lds_ptr || !tm->lds_voff)
    return error("prh_team_adjoint: null table");
  const int ncmax = (op->K + tm->nteam - 1) / tm->nteam;
  if (op->nsrc * ncmax > TTHREADS || op->nsrc * ncmax > WAVE * tm->coef_slots)
    return error("prh_team_adjoint: more source coefficients per team than staged");
  if (k_begin == k_end) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (int32_t e = refuse_capture(s)) return e;
  AdjArgs ta{*op, *sch, *adj, *tm, k_begin, k_end};
  const int nf = op->mvals_e ? 2 : 1;
  const void* fn = op->mvals_e ? reinterpret_cast<const void*>(&adjoint_march<true>)
                               : reinterpret_cast<const void*>(&adjoint_march<false>);
  return launch_march(fn, reinterpret_cast<const void*>(&adjoint_void), *tm,
                      (size_t)(TCONST + nf + 2 * tm->coef_slots + tm->lds_slots * nf),
                      &ta, s);
}
