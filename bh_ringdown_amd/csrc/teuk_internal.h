// Internal declarations shared by the libteuk host and device sources.
// Not part of the public C ABI (include/teuk.h).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <utility>
#include <vector>

#define TEUK_HD __host__ __device__ inline
#include "teuk_point.h"
#include "teuk_t4.h"

namespace teuk {

// parm.h:12 -- the 15-digit pi the reference uses for dtheta, cot and the
// spherical harmonics.
constexpr double kPi15 = 3.14159265358979;
// kern.cu:46
constexpr double kThird = 0.33333333333333333;
// kern.cu:196 -- first-derivative weight literal
constexpr double kD1 = 0.016666666666667;

// Stage-kernel tile: one wavefront owns 64 consecutive rho columns and a
// chunk of consecutive theta rows (theta_chunks); up to 4 wavefronts per
// block stack along theta.
constexpr int kWave = 64;
constexpr int kHalo = 4;            // KO reach in rho (kern.cu:247-256)
// Source patches are prepared for up to kRing steps per launch and kept in a
// ring of that many slots (step k uses slot k % kRing).
constexpr int kRing = 32;
constexpr int kLdsCols = kWave + 2 * kHalo;
// Whole-field sentinel: once per chunk of steps every field value is checked;
// a non-finite value, or a magnitude above this bound, marks the solve failed.
constexpr double kGrowthLimit = 1e60;

// Per-column constants of the coefficient fields (teuk_point.h).
using teuk_pt::kK1;
using teuk_pt::kK2;
using teuk_pt::kKA;
using teuk_pt::kKR;
using teuk_pt::kKD;
using teuk_pt::kKBt;
using teuk_pt::kKBr;
using teuk_pt::kKC0;
using teuk_pt::kKI0;
using teuk_pt::kKI1;
using teuk_pt::kKBi;
using teuk_pt::kKCi;
using teuk_pt::kNK;
// Per-row values: sin^2, cos, Y, tan(Pi/2 - theta); stored [4][M].
constexpr int kNR = 4;

// Scalar run description passed by value to every kernel.
struct Grid {
  int N, M;
  int even_m;          // ((int)m) % 2 == 0  (kern.cu:330)
  int ptsx, ptsy;
  int je;              // extraction column
  int Fr;
  int nrec_cap;        // output records the device buffers hold
  double xmin, xmax, dx, dtheta, dt;
  double mass, a, m;
  double start;
  int stag;            // 1: staggered second-order scheme (TD_GPU_code/Old);
                       // its source schedule holds two entries per step
};

// Gate of a resident launch (teuk_resident.inc): blocks that have arrived,
// and 0 undecided, 1 the launch runs, 2 it steps aside, changing nothing.
// Two per owner, used in turn: the finalize of a launch clears the other one.
struct ResGate {
  int arrived;
  int decision;
};

// How a solve's resident launches fared (written between them, k_finalize;
// the host sets it back).
struct ResTries {
  int fail;            // they have waited too long in a row: later ones do nothing
                       // until the host has run the missing steps
  int aside;           // launches in a row that stepped aside
  long long waited;    // ticks those waited
  int cur;             // segments: the fields are in 0 the state U, 1 the state D
  int asides;          // launches that stepped aside in all
};
// A launch's first wait before it steps aside, the waits in a row after which
// it is not tried again (ticks), and whether its steps change U and D's places.
struct ResTry {
  long long limit, budget;
  int flip;
};

// The most reads of a neighbour's flag in one wait, about a microsecond each.
constexpr int kResReads = 1 << 22;

// Device control block, one per solver.
struct Ctl {
  int k;               // completed steps
  int nrec;            // output records written
  int status;          // 0 ok; bit 0: non-finite Psi at the extraction column,
                       // bit 1: the whole-field sentinel fired (see kGrowthLimit),
                       // bit 2: a resident launch stopped half way (its fields are no state)
  ResTries tries;
  unsigned ended;      // blocks of the current record launch that have ended
  int reads;           // a resident launch's reads of a neighbour's flag in one wait (kResReads)
  double timer;        // solver time, advanced by repeated addition (body.cu:214)
  ResGate gate[2];
};

// Extraction state and output records (device pointers).
struct Ext {
  double *integ;       // [4][M] int Psi dt (re, im), int int Psi dt (re, im)
  double *snap;        // [nrec_cap][6][M] Psi, int, int int at output steps
  double *rec;         // [nrec_cap][16] t, dE/dt, h[14]
  int *rec_k;          // [nrec_cap][2] k, write flag
  const double *extw;  // [2M+1] dvol, rho2^4, rr^6 (body.cu:181-183)
  const double *projw; // [7][5*(M/4)][3] Boole/swsh factors per (l, term)
};

// Per-step particle scalars on the device (mirrors teuk_source_step).
struct SrcStep {
  double timer, start;
  double rp, tp, phip, E, lz, Q;
  double drdt, d2rdt2, dthdt, d2thdt2, dphidt, d2phidt2;
};

// One step of the source schedule on the device: canonical T_4 coefficients
// (filled by k_source_coeffs), particle position, radial Gaussian width,
// turn-on factor and the patch origin (kern.cu:1191-1206, 2673).
struct SrcDev {
  double c[12];
  double rp, tp, wr, turnon;
  int ip0, it0;
};

// Host-side preparation of one step (teuk_host.cpp).
struct SrcPrep {
  teuk_t4::StepIn in;
  SrcDev dev;
};

// Device pointers of one solver.
struct DevState {
  double *U, *C, *D, *A;   // field states (4 planes each); A only for RK4
  double *ktab;            // [kNK][N] column constants
  double *rtab;            // [kNR][M] row values
  double *dbdx;            // [M][N] rho derivative of bb (kern.cu:192-196)
  double *scratch;         // [M][N] set-up scratch (bb plane)
  double *theta, *r_c;     // [M], [N]
  double *phase;           // [2][N] cos, sin of the source phase (kern.cu:2671-2672)
  // Staggered scheme only: the half-point set (rho_a - dx/2, r_h).
  double *ktab_h;          // [kNK][N] column constants at the half points
  double *dbdx_h;          // [M][N] rho derivative of bb at the half points
  double *r_h;             // [N]
  double *phase_h;         // [2][N]
  double *patch;           // [kRing][2][ptsy][ptsx] source patches
  int *patch_org;          // [kRing][2] {row0, col0}
  SrcDev *sched;           // [nsched] source schedule, or null
  int nsched;
  Ext ext;
  Ctl *ctl;
};

// One member of a batch as the batched kernels see it: the run description,
// the solver's device pointers, its scheduled step count (steps at or past
// nt are skipped) and its tile count for the batch's block shape.
struct SolveDesc {
  Grid g;
  DevState d;
  int has_src;
  int ngroups;         // theta block-rows per rho strip
  int nt;
  int tiles;           // (N / 64) * ngroups
};

// One block's work in a batched stage launch: the member's description
// inline (one table read per block, not a tile entry and then a descriptor)
// and the tile within the member; tile < 0 pads the table.
struct BatchTile {
  SolveDesc sd;
  int tile;
  int pad[3];
};

// Resident stepping (teuk_resident.inc): B blocks of C rho columns each (the
// last may hold fewer), CP columns per thread.
constexpr int kResThreads = 512;
struct ResShape {
  int C, B, CP;
};
struct ResBlock {
  int member;          // index into the launch's descriptors
  int strip, C, B;     // block `strip` of the member's B blocks
};
// The columns [s0, s1) of a launch, those of them it stores ([v0, v1), into
// `out` from U, or from there into U where ResTries::cur says so), its plane for the coefficient values, the launch before it in the
// same steps (or null) and its first block's flags.
struct ResSpan {
  int s0, s1, v0, v1;
  double *out, *cpl;
  const ResGate *prev;
  int flag_blk;
};
// Column constants the resident kernel reads per stage, [N][8] (subset of kNK).
enum { kResA, kResBt, kResD, kResC0, kResI0, kResI1, kResBi, kResCi };
// The set-up plane (DevState::scratch, 8 N M >= 128 N bytes) holds after
// set-up the exchange flags ([blocks][32] words), the gates of segments' launches
// ([2][kMaxSegments], at the end of 16 N bytes) and the constants.
constexpr int kMaxSegments = 32;
TEUK_HD unsigned *res_flags(const DevState &d) { return reinterpret_cast<unsigned *>(d.scratch); }
TEUK_HD ResGate *res_gates(const DevState &d, int N) {
  return reinterpret_cast<ResGate *>(d.scratch + 2 * (size_t)N) - 2 * kMaxSegments;
}
TEUK_HD double *res_k8(const DevState &d, int N) { return d.scratch + 2 * (size_t)N; }
// The row count a kernel of CP columns per thread is built for: 0 any up to
// 64, kAnyTall any of 65 to 128 (two waves a column).
constexpr int kAnyTall = 1;
TEUK_HD constexpr int res_built_rows(int M, int CP) {
  if (CP < 4) return M == 64 || M == 32 ? M : 0;
  return M == 128 || M == 64 || M == 32 ? M : (M > kWave ? kAnyTall : 0);
}
// Groups of M threads in a block: any threads for the small-tile kernel (at
// least 8, one per edge column), within one or two waves each for the sweeping one.
TEUK_HD constexpr int res_groups(int M, int CP) {
  return CP >= 4 ? (M > kWave ? 4 : (kResThreads / kWave) * (kWave / M)) : (M > kWave ? 0 : kResThreads / M);
}
// Whether tiles of one column per thread exchange edge columns after every
// second stage only (0: no), and the columns per thread that the stage
// between then takes.
TEUK_HD constexpr int res_pair(int M, int C) {
  const int G = kResThreads / M;
  return C + 8 <= G ? 1 : (C <= G && G >= 16 ? 2 : 0);
}
// LDS of one block: columns of M + 1 rows of two complex fields (C + 16, twice;
// C + 12 for the sweeping kernel of CP >= 4), the extraction integrals, the column
// constants where they are not scalar loads.
TEUK_HD constexpr bool res_uniform(int M, int CP) { return CP > 4 && M >= kWave; }
TEUK_HD constexpr size_t res_lds_bytes(int M, int C, int CP) {
  return (size_t)(CP >= 4 ? 32 * (C + 12) : 64 * (C + 16)) * (M + 1) + 32 * (size_t)M +
         (CP >= 4 && !res_uniform(M, CP) ? 64 * (size_t)C : 0);
}
// The narrowest tile: a sweep reads the halo on its far side in its second
// phase, so no column of the first may reach it.
TEUK_HD constexpr int res_least_tile(int M, int CP) { return CP >= 4 ? ((res_groups(M, CP) * (CP / 2) + 11) & ~7) : 8; }
constexpr size_t kResLdsMax = 163840 - 512;   // a CU's LDS less the kernel's static part
constexpr int kResCP[5] = {1, 2, 4, 6, 8};
// Launches' longest wait in a row for all of their blocks to be on the GPU (s),
// unless one is given, and the longest taken: it must end in bounded time.
constexpr double kResWait = 0.25, kResWaitMost = 60.0;
// The first wait of a launch.  Two processes' launches that each hold CUs which
// the other waits for must not both wait on: one steps aside, the other runs,
// and the first's steps are taken by the launches queued behind it.  The wait
// is drawn from 0.5 to 1.5 times this, so that one is first, and doubles with
// each launch in a row that stepped aside, up to 6.4 ms, so that the launches
// of others (0.3 to 1.2 ms) are also waited out.  (A first wait of 0: the first
// try steps aside whatever happens, the next ones wait as others do.)
constexpr double kResPatience = 1e-4;
TEUK_HD long long res_patience(long long limit, int aside) {
  if (limit <= 0 && aside > 0) limit = 10000;
  const long long most = limit > 640000 ? limit : 640000;
  const long long w = limit << (aside < 20 ? aside : 20);
  return w < most ? w : most;
}
// That wait in the GPU's 100 MHz ticks; 0: it does not wait.
inline long long res_wait_ticks(double seconds) {
  if (!(seconds > 0.0)) return 0;
  return (long long)((seconds < kResWaitMost ? seconds : kResWaitMost) * 1e8) + 1;
}
// The wait of a launch that members with these waits share.
inline double res_shared_wait(const std::vector<double> &waits) {
  double w = kResWaitMost;
  for (double x : waits) w = x < w ? x : w;
  return w;
}
// The launch shape for an N x M grid on `cus` CUs, or false if its fields do
// not fit on the chip.
bool resident_shape(int N, int M, int cus, ResShape &sh);

// A grid that does not fit is stepped in segments of its columns, `steps`
// steps of one after the other: a segment's launch also computes the columns
// beside it that its steps reach (4 per stage), so segments need nothing from
// each other, and stores its own into a second state.  Empty: the per-stage
// kernels are faster, or the solve's buffers are too small for it.
struct ResSegments {
  int steps = 0;
  ResShape sh{0, 0, 0};             // of every segment (B: the widest)
  std::vector<ResSpan> spans;       // s0 .. v1 and flag_blk
};
ResSegments resident_segments(int N, int M, int integrator, int cus);

// Members of a batch that run in one resident launch: their tiles take at
// most one block per CU.
struct ResGroup {
  std::vector<int> members;   // indices into the shapes given
  std::vector<int> C;         // tile width of each
  int CP, MT;                 // columns per thread, the built-in M (0: any)
};
// The launches for members of the given N x M on `cus` CUs; a member whose
// fields do not fit on the chip is in none.
std::vector<ResGroup> resident_groups(const std::vector<std::pair<int, int>> &shapes, int cus);

// Theta chunks of one rho strip for wavefronts of R rows (R = 2, 4 or 8):
// the first chunk computes rows 3 .. 2+E and fills rows 0-2 from rows 3 and
// 4, the last computes rows M-3-E .. M-4 and fills M-3 .. M-1 from M-5 and
// M-4, and the rows between go R at a time.  E = edge_rows(R) >= 2 makes R
// divide what is left for every M that is a multiple of 8 and at least 16
// (the grids teuk_create accepts).
TEUK_HD constexpr int edge_rows(int R) { return R == 8 ? 5 : (R == 4 ? 3 : 2); }
TEUK_HD constexpr int theta_chunks(int M, int R) { return 2 + (M - 2 * edge_rows(R) - 6) / R; }
TEUK_HD constexpr bool theta_rows_ok(int M, int R) {
  return (R == 2 || R == 4 || R == 8) && M >= 16 && M % 8 == 0;
}
static_assert(theta_chunks(16, 8) == 2 && theta_chunks(64, 8) == 8 && theta_chunks(64, 4) == 15 &&
                  theta_chunks(64, 2) == 29 && theta_chunks(16, 2) == 5,
              "theta chunk layout");
// First row of theta chunk c, 0 <= c < theta_chunks(M, R): the first chunk
// starts at row 0, the last at theta_last_chunk_b0, chunk c in between at
// theta_inner_chunk_b0.  The edge chunks span edge_rows(R) + 3 rows (their
// computed rows and the three boundary rows), the others R.  (The stage
// kernel calls the per-kind forms inside its per-kind branches: a first row
// the compiler cannot see as 0 in the first chunk cost 15 % of the stage.)
TEUK_HD constexpr int theta_last_chunk_b0(int M, int R) { return M - edge_rows(R) - 3; }
TEUK_HD constexpr int theta_inner_chunk_b0(int R, int c) { return edge_rows(R) + 3 + (c - 1) * R; }
TEUK_HD constexpr int theta_chunk_b0(int M, int R, int c) {
  return c == 0 ? 0 : (c == theta_chunks(M, R) - 1 ? theta_last_chunk_b0(M, R) : theta_inner_chunk_b0(R, c));
}

// Block b of a single-solve stage launch of nblocks = S * ngroups blocks (S
// rho strips, ngroups block-rows per strip): its strip and block-row.  The
// hardware deals blocks round-robin over the 8 XCDs in dispatch order; each
// XCD gets a contiguous run of tiles, so the halos its waves re-read stay in
// its own L2.  edge_first: XCD x owns strips [x S/8, (x+1) S/8) when the
// strips split evenly, and the block-rows holding a strip's first and last
// theta chunk are dispatched before the others.
TEUK_HD void stage_block_tile(int b, int nblocks, int ngroups, bool edge_first, int &strip, int &grp) {
  if (!edge_first) {
    int tile = b;
    if ((nblocks & 7) == 0) tile = (b & 7) * (nblocks >> 3) + (b >> 3);
    strip = tile / ngroups;
    grp = tile - strip * ngroups;
    return;
  }
  const int S = nblocks / ngroups;
  int j = b, s0 = 0, ns = S;
  if ((S & 7) == 0) {
    ns = S >> 3;
    s0 = (b & 7) * ns;
    j = b >> 3;
  }
  const int ne = ngroups >= 2 ? 2 : 1;   // edge block-rows per strip
  if (j < ne * ns) {
    strip = s0 + j / ne;
    grp = (j % ne) ? ngroups - 1 : 0;
  } else {
    const int jj = j - ne * ns;
    strip = s0 + jj / (ngroups - 2);
    grp = 1 + jj % (ngroups - 2);
  }
}
constexpr int kDefaultThetaRows = 2;
constexpr int kDefaultWavesPerEU = 2;   // a batch's until set (teuk_batch_set_tiling)

// Stage-kernel launch shape: wavefronts per block (1, 2 or 4), the
// occupancy hint the kernel was compiled for (waves per SIMD: 2 or 4) and
// the theta rows per wavefront (2, 4 or 8).
struct Tiling {
  int wpb;
  int wpe;
  int rows;
};

// Launchers (teuk_kernels.hip).
hipError_t launch_init_coeffs(const Grid &g, const DevState &d, hipStream_t s);
hipError_t launch_source_coeffs(const teuk_t4::StepIn *in, SrcDev *sched, int n, hipStream_t s);
// Patches of n <= kRing consecutive steps from (step counter + k_rel0).
// colmajor: patches stored column after column (the resident kernel's lanes
// run along theta), else row after row.
hipError_t launch_source(const Grid &g, const DevState &d, int k_rel0, int n, bool colmajor, hipStream_t s);
// The patch of absolute step kstep (into its ring slot).
hipError_t launch_source_at(const Grid &g, const DevState &d, int kstep, hipStream_t s);
hipError_t launch_stage(const Grid &g, const DevState &d, int integrator, int stage,
                        bool has_src, int k_rel, Tiling t, hipStream_t s);
// gate: the gate of the resident launch that ran the steps (the other of its
// pair, or all `others` of it, is cleared) and what it waited, or null.
hipError_t launch_finalize(const Grid &g, const DevState &d, int n, ResGate *gate, ResGate *other, ResTry t,
                           hipStream_t s, int others = 1);
// The ABI's four real planes to the device's two planes of pairs and back
// (in and out apart).
hipError_t launch_fields_join(const double *in, double *out, size_t NM, hipStream_t s);
hipError_t launch_fields_split(const double *in, double *out, size_t NM, hipStream_t s);
// Flags and column constants of resident stepping, into the set-up plane.
hipError_t launch_init_res(const Grid &g, const DevState &d, hipStream_t s);
// nsteps <= kRing steps of one solve (at most to step nt) in one launch.
hipError_t launch_resident(const Grid &g, const DevState &d, int integrator, bool has_src, ResShape sh,
                           const ResSpan &sp, int nsteps, int nt, ResGate *gate, long long limit, hipStream_t s);
// The same for the blocks of several solves (a group of resident_groups), each
// at most to its own last step; lds: the largest member's res_lds_bytes.
hipError_t launch_resident_batch(const SolveDesc *descs, const ResBlock *blocks, int nblocks, int integrator, int CP,
                                 int MT, size_t lds, int nsteps, ResGate *gate, long long limit, hipStream_t s);
template <int CP>
hipError_t launch_resident_batch_cp(const SolveDesc *descs, const ResBlock *blocks, int nblocks, int integrator, int MT,
                                    size_t lds, int nsteps, ResGate *gate, long long limit, hipStream_t s);
template <int CP>
hipError_t launch_resident_cp(const Grid &g, const DevState &d, int integrator, bool has_src, ResShape sh,
                              const ResSpan &sp, int nsteps, int nt, ResGate *gate, long long limit, hipStream_t s);
// The whole-field sentinel over the current fields (state U); enqueued once
// per chunk of steps, before the chunk's launch_finalize.
hipError_t launch_sentinel(const Grid &g, const DevState &d, hipStream_t s);
// Staggered second-order scheme (teuk_so2.hip): bb and dbdx of both point
// sets, and one step (half step, its theta edges, full step, edges and
// extraction).
hipError_t launch_init_so2(const Grid &g, const DevState &d, hipStream_t s);
hipError_t launch_so2_step(const Grid &g, const DevState &d, bool has_src, int k_rel, hipStream_t s);
// Batched forms: one launch covers every member of the batch.
hipError_t launch_source_batch(const SolveDesc *descs, int nsolves, int max_cells, int k_rel0, int n,
                               bool colmajor, hipStream_t s);
hipError_t launch_stage_batch(const BatchTile *tiles, int ntiles, int integrator, int stage, int k_rel, Tiling t,
                              hipStream_t s);
// The stage builds for R theta rows per wavefront (teuk_stage_r<R>.hip),
// behind launch_stage / launch_stage_batch.
template <int R>
hipError_t launch_stage_rows(const Grid &g, const DevState &d, int integrator, int stage, bool has_src, int k_rel,
                             int ngroups, dim3 grid, dim3 block, int wpe, hipStream_t s);
template <int R>
hipError_t launch_stage_batch_rows(const BatchTile *tiles, int ntiles, int integrator, int stage, int k_rel,
                                   dim3 block, int wpe, hipStream_t s);
hipError_t launch_finalize_batch(const SolveDesc *descs, int nsolves, int n, ResGate *gate, ResGate *other, ResTry t,
                                 hipStream_t s);
// The sentinel of every member still running before the chunk's finalize.
hipError_t launch_sentinel_batch(const SolveDesc *descs, int nsolves, hipStream_t s);
// Default launch shape for an N x M grid.
Tiling default_tiling(int N, int M);
// Blocks per rho strip for wpb waves per block of `rows` theta rows each
// (the last may hold surplus waves, which return at once).
int stage_groups(int M, int wpb, int rows);
bool source_available();

// Host helpers (teuk_host.cpp).
void host_grid(int N, int M, double xmin, double xmax, double mass, double a,
               double *x_c, double *r_c, double *theta);
// Half points of the staggered scheme: rho_h = xmin + (l - 1/2) dx, r_h(rho_h).
void host_grid_half(int N, double xmin, double xmax, double mass, double a, double *x_h, double *r_h);
double host_swsh(double ell, double ml, double the);
void host_projection_weights(int M, double m, double *w /*[7][5*(M/4)][3]*/);
// Column constants [kNK][N] at rho = xmin + (j + shift) dx with radius r[j]
// and row values [kNR][M] of the coefficient fields; `staggered` selects the
// staggered scheme's cot (cos/sin, Old/kern.cu:241-243) for the last row value.
void host_coeff_tables(int N, int M, double xmin, double xmax, double dx, double mass, double a,
                       double m, const double *r, const double *theta, double *ktab,
                       double *rtab, double shift = 0.0, bool staggered = false);
// Source phase e^{-i m a ln((r-r+)/(r-r-))/(r+-r-)} per column, [2][N].
void host_source_phase(int N, double mass, double a, double m, const double *r_c, double *phase);
// Per-step transcendentals and patch placement of the source (kern.cu:1186-1206, 2673).
void host_source_prepare(const Grid &g, const SrcStep &st, SrcPrep &out);

}  // namespace teuk
