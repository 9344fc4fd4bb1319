// Internal data model of the MI355X Fock build (host + device).
//
// The reference keeps, per pair class, arrays of primitive-pair data behind
// CSR offsets (shell_pair_t, src/liberi_types.f90:80-92) and rebuilds the
// screened pair lists on the host for every kernel call
// (e.g. src/rhf/rot_axis/int0001.F90:65-84).  Here every shell pair of every
// class lives once in HBM as a fixed-size record, every primitive pair as a
// 64-byte record, and each of the 55 classes owns its screened, sorted pair
// lists plus a segment table that enumerates the surviving quartets without
// materialising them.
#pragma once

#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

namespace liberi {

constexpr int kNumClasses = 55;
constexpr int kNumPairClasses = 10;
constexpr double kRefCutoff = 5.00000000000000018e-11;  // src/liberi_parameters.F90:38
constexpr double kTwoPi52 = 34.98683665524971863;        // 2 pi^(5/2), :20

// pair classes in the order of shell_pair_container_t (src/liberi_types.f90:94-109)
enum PairClass { P_SS, P_SP, P_PP, P_SD, P_PD, P_DD, P_SF, P_PF, P_DF, P_FF };
constexpr int kPairL[kNumPairClasses][2] = {{0, 0}, {0, 1}, {1, 1}, {0, 2}, {1, 2},
                                            {2, 2}, {0, 3}, {1, 3}, {2, 3}, {3, 3}};

enum QuartetTest { CMP_GT, CMP_GE, CMP_NONE };
enum PreScreen { PS_CROSS, PS_SELF };

struct ClassDef {
  const char *name;
  int bra, ket;  // pair classes; bra == ket marks a diagonal class (kl <= ij)
  int cmp, ps;
};

// Dispatch order of src/liberi_driver.F90:69-158.  Quartet test and pair
// pre-screen per kernel file: the hand-written rotated-axis kernels normalise
// each list's pre-screen by the OTHER list's largest Schwarz value
// (int0001.F90:67,76), the generated Rys/ERIC kernels by their own
// (int3300_rysgen.F90, int0030_ericgen.F90); int0000/int0101/int1111 skip when
// x*x < cut (int0000.F90:107), int2222gen and int3333 have no quartet test
// (int2222_rysgen.F90:428-431), every other kernel keeps x*x > cut.
extern const ClassDef kClasses[kNumClasses];

// One shell pair, A = the shell of higher angular momentum (A first for equal L).
struct PairRec {
  int32_t prim_off;  // first primitive pair record (the k-th is prim_stride k further on)
  int32_t nprim;
  int32_t bfA, bfB;  // first basis function (0-based) of A and B
  double ABx, ABy, ABz;
  int32_t sameAB;    // A and B are one shell
  int32_t prim_stride;  // primitive record k is prims[prim_off + k * prim_stride]
  int32_t cA, cB;    // compact column of A's / B's first function among all
                     // functions of that angular momentum (shell rank * ncart)
  double x;          // Schwarz value of the pair
};

// largest basis: n(n+1) stays below 2^32, so packed indices fit 32 bits
constexpr int32_t kMaxBasis = 65535;

// One primitive pair (a in A, b in B): p = a + b, P, P - A, and
// K = c_a c_b exp(-ab/p |A-B|^2) / p.
struct alignas(64) PrimRec {
  double p, Px, Py, Pz, PAx, PAy, PAz, K;
};

// One workgroup of a row-tiled kernel: the quartets [q0, q0 + n) of one row,
// in the segments seg to last; in the lane-per-quartet kernels `team` adjacent
// lanes share a quartet (a power of two up to 64).
struct RowTile {
  int64_t q0;
  int32_t n, seg, team, last;
};

// workgroup sizes of the lane row-tiled kernels
constexpr int kRowThreads[2] = {256, 512};

// Device view of one class's quartet enumeration.  Kept pair lists are sorted
// by (primitive count, Schwarz value descending); a segment is one kept bra
// row against one primitive-count group of kets, and its surviving kets are a
// prefix of that group (the quartet test is monotone in the ket's Schwarz
// value).  Quartet q of the class lies in segment s with
// seg_start[s] <= q < seg_start[s+1], ket = seg_ket0[s] + q - seg_start[s]: the
// PairRec array itself is in that order, so that the kets of a segment, and
// their k-th primitive records, are neighbours in memory.
struct ClassDev {
  const int64_t *seg_start;  // nseg + 1
  const int32_t *seg_bra;    // bra pair index of the segment
  const int32_t *seg_ket0;   // ket pair index of the segment's first quartet
  int32_t nseg;
  int32_t diag;
  int64_t q_begin, q_end;    // this rank's share of the class's quartets
  double xswitch;            // Rys argument from which the asymptotic rule is used
  // this rank's row tiles in launch order; row_mode selects the row-tiled kernel
  const RowTile *tiles;
  int32_t ntile;
  int32_t row_mode;
  int32_t threads;  // of a workgroup of the lane row-tiled kernel
  // 0: rows run over the class's bra pairs, segments over its kets (as
  // above); 1: the roles are swapped -- seg_bra holds ket pairs and seg_ket0
  // bra pairs -- so that a row tile fixes the ket pair (non-diagonal classes)
  int32_t transposed;
  // the fixed (rows) and the moving pairs' classes in the pair layout: element
  // of component k of pair p is base + k * n + p
  int64_t fix_base, mov_base;
  int32_t fix_n, mov_n;
  // the bra and the ket pairs' classes in the pair-major form: element of
  // component k of pair p is bra_q + p * components + k
  int64_t bra_q, ket_q;
  // group and cooperative kernels: chunk_stride(grid) of the launch (set at launch)
  int64_t chunk_stride;
  // 1: the mixed form may evaluate this class's quartets in FP32 (chosen per
  // class at the first build under a given switch tau)
  int32_t fp32;
  // 1: a class with a cooperative form (class_has_coop) runs that form
  int32_t coop;
};

// Pair layout: quantities with one value per (shell pair, component pair) of
// every pair class, class after class, component-major over the class's pairs
// in device order, components a * nb + b in internal order.  The element of
// component k of pair p of class c is off[c] + k * n[c] + (p - first[c]), so
// consecutive pairs are neighbours in memory: the Coulomb sums of a row
// tile's moving pairs are added there instead of to F, 64 lanes to 64
// consecutive doubles (measured 187 G atomic adds/s against 23.7 G to
// scattered ones).  The pair-major form has component k of pair p at
// off[c] + (p - first[c]) * components + k.
struct PairLayout {
  int64_t off[kNumPairClasses + 1];
  int32_t n[kNumPairClasses], first[kNumPairClasses];
  // workgroups of the kernels over it: those of class c are [block[c],
  // block[c + 1]), chunks[c] per component
  int32_t chunks[kNumPairClasses], block[kNumPairClasses + 1];
};

// the densities of BuildArgs the start of a build fills
struct BuildWork {
  double *Dp, *Dq, *Dsq;
};

struct BuildArgs {
  const PairRec *pairs;
  const PrimRec *prims;
  const double *D;   // density of the Coulomb blocks (packed)
  const double *DK;  // density of the exchange blocks (= D for RHF, packed)
  const double *Dp, *Dq;  // D in the pair layout, component- and pair-major
  const double *Dsq;  // DK as a full nbf x nbf matrix
  // sums that the end of the build adds to F: Coulomb blocks in the pair
  // layout, component-major (kernels with a pair per lane) and pair-major
  // (kernels with a pair's components over the lanes), and exchange blocks as a
  // full matrix, rows the functions of one pair and columns those of the
  // other, so that a block's rows are runs of consecutive elements
  double *Jp, *Jq, *Ksq;
  double k_scale;    // exchange weight (1 for RHF: F = J[D] - K[D]/2; 2 for a UHF spin: J[Da+Db] - K[Ds])
  double *F;
  double value_cut;
  int32_t nbf;           // basis functions
  // compact columns of the row-tiled accumulators: the functions of angular
  // momentum L in shell order, col_bf[L][k] = basis function of column k
  const int32_t *col_bf[4];
  int32_t ncol[4];
  // mixed precision: quartets with x_bra * x_ket * dmax[0] < fp32_tau in FP32
  double fp32_tau;
  const double *dmax;        // max |D| of this build (device)
  uint64_t *fp32_count;      // quartets evaluated in FP32 (device counter)
};

// Launch the kernel of class c over [q_begin, q_end).  Returns hipError_t.
int launch_class(int c, const ClassDev &cd, const BuildArgs &ba, void *stream, int num_wg_coop);
// 1 when group class c has the wave-split row-tiled form (its row form)
int class_has_split(int c);
// kernel attributes the launches of class c need (the wave-split kernels'
// dynamic LDS above 64 KB), on the current device; called at setup, outside
// any stream capture.  Returns hipError_t.
int prepare_class(int c);
// Rys roots of class c and the end of its tabulated range
int class_nroots(int c);
double class_rys_xmax(int c);
// LDS bytes of the row-tiled kernel of class c with rows over the bra pairs
// (transposed = 0) or the ket pairs (1), given the compact column counts per
// angular momentum and the Rys switch (the kernel stages the table below it);
// -1 when the class has no such kernel
int64_t class_row_lds(int c, int transposed, const int32_t *ncol, double xswitch);
// quartets a workgroup of the class's row-tiled kernel holds at one lane each
int class_row_quartets(int c);
// longest chain of primitive quartets a lane of class c is left with in a
// share of primq primitive quartets (0: the class's kernel has no teams)
double class_row_chain(int c, int64_t primq);
// kernel shape of class c: 0 lane per quartet, 1 workgroup group per
// quartet, 2 cooperative workgroup per quartet
int class_kernel_kind(int c);
// 1 when class c also has the cooperative form ((dd|dd), (fs|fs) and the group
// classes with an f shell), selected by ClassDev::coop
int class_has_coop(int c);

// Fused group launch: one work item = quartets [c0, c1) of class cls (relative
// to the class's share, c0 a multiple of its quartets per round)
struct FusedItem {
  int32_t cls, pad;
  int64_t c0, c1;
};
// quartets per round of class c in the fused group launch (0: not fused)
int class_fused_nq(int c);
// the items[0 .. nitems) of the build, taken through the counter *head
// (zero before the launch); cds: ClassDev of every class by class index
int launch_group_fused(const ClassDev *cds, const BuildArgs &ba, const FusedItem *items, int64_t nitems,
                       unsigned long long *head, int nwg, void *stream);
// Shared launches: the workgroups of several small classes in one launch.
// Entry k is class cls[k] with the workgroups [first[k], first[k + 1]).
constexpr int kSharedLaunches = 6;
struct SharedArgs {
  int32_t n = 0, lds = 0;  // entries; dynamic LDS bytes (row-tiled launches)
  int32_t cls[18], first[19];
};
// shared launch that has a body of class c (in that orientation of its rows),
// or -1; launches below kSharedRowLaunches run the row-tiled form with
// kSharedRowThreads threads, the group launch the group form, the others the
// cooperative one
constexpr int kSharedRowLaunches = 3, kSharedGroupLaunch = 3, kSharedRowThreads = 256;
int class_shared_launch(int c, int transposed);
// quartets per round of a workgroup of class c in its (group or cooperative) shared launch
int class_round_quartets(int c);
int launch_shared(int launch, const SharedArgs &sa, const ClassDev *cds, const BuildArgs &ba, void *stream);

// row-tile lengths (quartets of one row per workgroup) the autotuner times
// per row-tiled class; kDefaultTile where it does not time
constexpr int kNumTileLens = 4;
constexpr int64_t kTileLens[kNumTileLens] = {512, 1024, 4096, 16384};
constexpr int kDefaultTile = 2;
// Spreading a class over the chip.  A lane evaluates a quartet's primitive
// quartets one after the other, up to 1296 in (ss|ss), 0.1 to 2 us each, so a
// class of few quartets is bound by its longest chain (water's (ss|ss): 406
// quartets, 0.30 ms).  `team` lanes then share a quartet: each takes every
// team-th primitive of the moving pair.  A team costs the wave its fixed work
// (records, the sum over the team, the digestion, which one lane does) for
// 64 / team quartets, d primitive quartets' worth; with C the longest chain
// left to a lane, a class of p primitive quartets on the waves the chip runs
// at once takes about (p / C) d / (64 kRowWaves) + C, least at
// C = sqrt(p d / (64 kRowWaves)).  Measured on 12 atoms of the cage: (ss|ss)
// 0.39 -> 0.10 ms, (ss|ps) 0.28 -> 0.11; on water 0.30 -> 0.02, 0.20 -> 0.02.
constexpr double kRowWaves = 1740;  // 1024 SIMDs, 1.7 waves each
// a class of at most this many workgroup steps runs one step per tile: its
// tiles then still fit the chip a few times over, and the flush of a tile's
// exchange rows costs less than the idle compute units (more steps: the timed
// tile length; C60's (dd|dp), 9100 steps on 1830 rows, 5.1 ms in whole rows,
// 6.1 cut to steps)
constexpr int64_t kRowSteps = 1024;
// LDS the row-tiled kernel may take per workgroup
constexpr int64_t kRowLdsBytes = 64 * 1024;
// workgroups the cooperative kernels use at most
constexpr int kCoopWorkgroups = 8192;
// one-wave workgroups the group-per-quartet kernels use at most (persistent loop)
constexpr int kGroupWorkgroups = 65536;

// Order in which the workgroups of a persistent group-kernel launch take the
// contiguous chunks of a class's quartet range: workgroup b takes chunk
// b * s mod grid.  The stride s is coprime with the grid, so the map is a
// permutation of 0 .. grid-1 for every grid size, and close to grid divided by
// the golden ratio, so that workgroups resident at the same time (consecutive
// b) work on distant parts of the range.
constexpr int64_t chunk_stride(int64_t grid) {
  if (grid <= 2) return 1;
  int64_t s = (int64_t)((double)grid * 0.6180339887498949) | 1;
  for (;; ++s) {  // ends at the latest at s = grid - 1, coprime with grid
    int64_t a = grid, b = s;
    while (b != 0) {
      const int64_t t = a % b;
      a = b;
      b = t;
    }
    if (a == 1) return s;
  }
}

// Schwarz integrals of a whole basis.  The host stages the shells and the
// list of shell pairs; the primitive-pair records are formed on the device.
struct SchwarzShell {
  double x, y, z;
  int32_t first, k;  // its exponents and coefficients in SchwarzStage::ew
};
// one shell pair, A the shell of higher angular momentum
struct SchwarzPair {
  int32_t a, b;            // shells
  int32_t prim_off, nprim;  // its primitive records
};
// every shell pair i >= j, grouped by (la, lb) (group la*4+lb is
// pairs[off[k] .. off[k+1])), per pair its packed index i(i+1)/2 + j, and the
// longest primitive list of each group
struct SchwarzStage {
  std::vector<SchwarzShell> shells;
  std::vector<double> ew;  // exponents of all shells, then their coefficients
  std::vector<SchwarzPair> pairs;
  std::vector<int64_t> where;
  int64_t nprims = 0;
  size_t off[17];
  int32_t longest[16];
  // byte offsets of the parts of the device buffer -- the stage (`upload`
  // bytes in one copy: pairs | shells | ew), primitive records, results -- and
  // its size
  size_t o_shells, o_ew, upload, o_prims, o_out, bytes;
};
// the primitive-pair records of the staged pairs
int launch_schwarz_records(const SchwarzPair *pairs, int32_t n, const SchwarzShell *shells, const double *ew,
                           int32_t nprim_total, PrimRec *prims, void *stream);
// Schwarz values sqrt(max |(ab|ab)|) of the n shell pairs `pairs`, whose
// shells have angular momenta la >= lb and at most `longest` primitive pairs;
// out[i] for pairs[i].
int launch_schwarz(int la, int lb, const SchwarzPair *pairs, const SchwarzShell *shells, const PrimRec *prims,
                   int32_t n, int32_t longest, double *out, void *stream);
// checked basis -> stage (LIBERI_OK or a status with the message set)
int schwarz_stage(const char *who, int32_t nsh, int32_t natoms, int32_t num_bas, int32_t mxgtot,
                  const int32_t *ang_mom, const int32_t *contr_num, const int32_t *sh_loc, const int32_t *atom_num,
                  const int32_t *atom_loc, const double *exponents, const double *cs, const double *cp,
                  const double *cd, const double *cf, const double *coords, SchwarzStage &s);
// a gfx950 device is current (LIBERI_OK or LIBERI_EDEVICE with the message set)
int schwarz_check_device(const char *who);
// the stage uploaded to the device buffer `buf` (s.bytes, 256-byte aligned) and
// the kernels that leave the results at s.o_out (pair order); `host` receives
// the upload and has to live until the stream has been waited for; returns a
// hipError_t
int schwarz_enqueue(const SchwarzStage &s, unsigned char *buf, std::vector<unsigned char> &host, void *stream);
// out (pair order) -> schwrz_int (packed by shell pair)
void schwarz_scatter(const SchwarzStage &s, const double *out, double *schwrz_int);
// records the message of liberi_c_last_error and returns code
int set_last_error(int code, const std::string &msg);

// start of a build (F and the sums zeroed, Dp, Dq and Dsq filled from D and
// DK) and its end (the sums added to F)
int launch_build_begin(const BuildArgs &ba, const PairLayout &pl, const BuildWork &w, void *stream);
int launch_build_end(const BuildArgs &ba, const PairLayout &pl, void *stream);

// p[0..n) = 0 on the stream (a kernel, so it may sit in a captured graph)
int launch_fill_zero(double *p, int64_t n, void *stream);
// out = a + b over n elements
int launch_add(const double *a, const double *b, double *out, int64_t n, void *stream);
// out[0] = max |p[0..n)| (out must be zero on entry)
int launch_abs_max(const double *p, int64_t n, double *out, void *stream);

// Segment lengths on the device: one thread per (kept bra row, ket group) of
// every job (a class), job j in the workgroups from block0 on.  The arrays are
// byte offsets from `base`; bra_group is read in diagonal classes only, whose
// bras and kets are one list.
constexpr int kSegThreads = 256;
struct SegJob {
  int64_t bra_x, bra_group, ket_x, group_begin, group_end;  // byte offsets
  int64_t len0, block0;
  int32_t nbra, ngroup, diag, cmp;
};
int launch_segment_lengths(const unsigned char *base, const SegJob *jobs, int32_t njob, int64_t nblock, double cut,
                           int32_t *seg_len, void *stream);

}  // namespace liberi
