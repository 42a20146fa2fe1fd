// HIP kernels of libteuk other than the Runge-Kutta stage (teuk_stage.inc):
// the time-independent coefficient planes, the particle-source patches, the
// output records and the whole-field sentinel, and the launchers of all of
// them, the stage included (launch_stage picks the stage build for the
// launch shape's theta rows).
#include "teuk_dev.h"

namespace teuk {
namespace {


// ---------------------------------------------------------------------------
// bb on interior rows (kern.cu:147) into a scratch plane, then its 6th-order
// rho derivative (kern.cu:192-196), which is time independent.
__global__ __launch_bounds__(256) void k_init_bb(Grid g, const double *__restrict__ ktab,
                                                 const double *__restrict__ rtab, double *__restrict__ bbp) {
  const size_t NM = (size_t)g.N * g.M;
  const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= NM) return;
  const int k = (int)(id / g.N), j = (int)(id - (size_t)k * g.N);
  double bb = 0.0;
  if (k >= 3 && k < g.M - 3) {
    double K[kNK];
#pragma unroll
    for (int i = 0; i < kNK; i++) K[i] = ktab[(size_t)i * g.N + j];
    bb = coef_point(K, rtab[k], rtab[g.M + k], rtab[2 * g.M + k]).bb;
  }
  bbp[id] = bb;
}

__global__ __launch_bounds__(256) void k_init_dbdx(Grid g, const double *__restrict__ bbp,
                                                   double *__restrict__ dbdx) {
  const size_t NM = (size_t)g.N * g.M;
  const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= NM) return;
  const int a = (int)(id % g.N);
  double d = 0.0;
  if (a >= 3 && a < g.N - 3)
    d = teuk_pt::d1(bbp[id + 1], bbp[id - 1], bbp[id + 2], bbp[id - 2], bbp[id + 3], bbp[id - 3],
                    kD1 * (1.0 / g.dx));
  dbdx[id] = d;
}


// ---------------------------------------------------------------------------
// What resident stepping keeps in the set-up plane once dbdx is formed: its
// exchange flags, cleared, and the column constants it reads, [N][8].
__global__ __launch_bounds__(256) void k_init_res(Grid g, DevState d) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= g.N) return;
  unsigned *flags = res_flags(d);
  for (int i = 0; i < 4; i++) flags[4 * (size_t)j + i] = 0;
  constexpr int src[8] = {kKA, kKBt, kKD, kKC0, kKI0, kKI1, kKBi, kKCi};
#pragma unroll
  for (int i = 0; i < 8; i++) res_k8(d, g.N)[(size_t)j * 8 + i] = d.ktab[(size_t)src[i] * g.N + j];
}

// The ABI's four real planes (q_re, q_im, p_re, p_im) to the device's two
// planes of (re, im) pairs, and back.  The host's copy bounds both: 268 MB
// (65536 x 128) cross the bus in 9.5 ms and take 0.1 ms here, where
// interleaving them in host memory first took 59 ms.
__global__ __launch_bounds__(256) void k_fields_join(const double *__restrict__ in, double *__restrict__ out,
                                                     size_t NM) {
  for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < 2 * NM; c += (size_t)gridDim.x * blockDim.x) {
    const size_t h = c >= NM ? NM : 0;   // plane base: 0, NM of the pairs, twice that of the reals
    reinterpret_cast<double2 *>(out)[c] = make_double2(in[c + h], in[c + h + NM]);
  }
}

__global__ __launch_bounds__(256) void k_fields_split(const double *__restrict__ in, double *__restrict__ out,
                                                      size_t NM) {
  for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < 2 * NM; c += (size_t)gridDim.x * blockDim.x) {
    const size_t h = c >= NM ? NM : 0;
    const double2 v = reinterpret_cast<const double2 *>(in)[c];
    out[c + h] = v.x;
    out[c + h + NM] = v.y;
  }
}

// Output records for a batch of n completed steps (body.cu:174-212): for each
// step k with k % Fr == 0, the energy flux from the snapshot of int Psi dt
// and the 14 projections of int int Psi dt onto -2Y_lm (proj.c:37-75); the
// solver time advanced by repeated addition (body.cu:214).  Explicit
// round-to-nearest operations in the reference's evaluation order make the
// records equal the host computation bit for bit.  Then advances the step
// counter by n.
//
// One block per record: latency bounds it (a record is 15 sums of M to 5 M/4
// terms).  The threads form the terms side by side, kFinTerms per sum at a
// time, into LDS; 15 threads then add them up in order.  [term][sum] keeps
// the adders' reads free of bank conflicts.  The block that ends last
// advances the counters, which every block reads when it starts.  32 records
// of 64 rows: 24.8 us with one block and one thread per sum, now 6.2 us;
// of 128 rows (16 records) 36.3, now 8.5.
constexpr int kFinTerms = 80;
constexpr int kFinThreads = 512;

__device__ __forceinline__ void finalize_solve(const Grid &g, const Ext &ext_in, Ctl *ctl_in, int n,
                                               const ResGate *gate, ResGate *other, int others, const ResTry &tr,
                                               int first) {
  __shared__ double terms[kFinTerms][15];
  const int M = g.M, t = threadIdx.x;
  if (gate) {
    if (first && t < others) other[t].arrived = other[t].decision = 0;
    // the launch stepped aside, or did nothing as an earlier one's waits were
    // too long: no step was taken
    if (gate->decision != 1) {
      if (first && t == 0) {
        ResTries &r = ctl_in->tries;
        r.waited += res_patience(tr.limit, r.aside);
        r.aside++;
        r.asides++;
        if (r.waited >= tr.budget) r.fail = 1;
      }
      return;
    }
  }
  // global-memory views of the solve's buffers (see global_ptr)
  struct {
    const TEUK_GLOBAL double *snap, *extw, *projw;
    TEUK_GLOBAL double *rec;
    TEUK_GLOBAL int *rec_k;
  } ext = {global_ptr(const_cast<const double *>(ext_in.snap)), global_ptr(ext_in.extw), global_ptr(ext_in.projw),
           global_ptr(ext_in.rec), global_ptr(ext_in.rec_k)};
  TEUK_GLOBAL Ctl *ctl = global_ptr(ctl_in);
  const int k0 = ctl->k;
  const double timer0 = ctl->timer;
  const int r_lo = (k0 + g.Fr - 1) / g.Fr;                 // first record in [k0, k0+n)
  int r_hi = (k0 + n - 1) / g.Fr + 1;                       // one past the last
  if (r_hi > g.nrec_cap) r_hi = g.nrec_cap;
  const double dt = g.dt;
  const int nterm = 5 * (M / 4);
  for (int r = r_lo + blockIdx.x; r < r_hi; r += gridDim.x) {
    const TEUK_GLOBAL double *sn = ext.snap + (size_t)r * 6 * M;
    TEUK_GLOBAL double *rec = ext.rec + (size_t)r * 16;
    const double r6 = ext.extw[2 * M];
    double sum = 0.0;
    for (int lo = 0; lo < nterm; lo += kFinTerms) {
      const int cnt = nterm - lo < kFinTerms ? nterm - lo : kFinTerms;
      // the 14 projections' terms: Boole group i / 5 covers rows 4 (i / 5) .. 4 (i / 5) + 4
      for (int task = t; task < 7 * cnt; task += kFinThreads) {
        const int l = task / cnt, i = lo + task % cnt;
        const TEUK_GLOBAL double *w = ext.projw + ((size_t)l * nterm + i) * 3;
        const int pt = 4 * (i / 5) + i % 5, row = pt < M ? pt : M - 1;
        const double w0 = w[0], w1 = w[1], w2 = w[2], re = sn[4 * M + row], im = sn[5 * M + row];
        terms[i - lo][2 * l] = __dmul_rn(__dmul_rn(__dmul_rn(__dmul_rn(w0, re), w1), g.dtheta), w2);
        terms[i - lo][2 * l + 1] = __dmul_rn(__dmul_rn(__dmul_rn(__dmul_rn(w0, im), w1), g.dtheta), w2);
      }
      // the flux's terms, one per row
      for (int q = lo + t; q < lo + cnt && q < M; q += kFinThreads) {
        const double ir = sn[2 * M + q], ii = sn[3 * M + q];
        const double psi2 = __dadd_rn(__dmul_rn(ir, ir), __dmul_rn(ii, ii));
        terms[q - lo][14] = __ddiv_rn(__dmul_rn(__dmul_rn(psi2, ext.extw[q]), r6), ext.extw[M + q]);
      }
      __syncthreads();
      if (t < 15) {
        const int upto = t == 14 ? (M - lo < cnt ? M - lo : cnt) : cnt;
#pragma unroll 8
        for (int i = 0; i < upto; i++) sum = __dadd_rn(sum, terms[i][t]);
      }
      __syncthreads();
    }
    if (t < 14) {
      const double h = __ddiv_rn(__dmul_rn(2.0, sum), 45.0);
      rec[2 + t] = (t & 1) ? -h : h;
    } else if (t == 14) {
      const int k = r * g.Fr;
      double timer = timer0;
      for (int i = k0; i < k; i++) timer = __dadd_rn(timer, dt);
      rec[0] = timer;
      rec[1] = sum;
      ext.rec_k[2 * r] = k;
      ext.rec_k[2 * r + 1] = ((double)k * dt) >= (g.xmax + 200.0) ? 1 : 0;
    }
  }
  // the last block to end advances the counters: all threads have read them
  __syncthreads();
  if (t == 0 && atomicAdd(&ctl_in->ended, 1u) + 1 == gridDim.x) {
    double timer = timer0;
    for (int i = 0; i < n; i++) timer = __dadd_rn(timer, dt);
    ctl->ended = 0;
    if (gate) {
      ctl->tries.aside = 0;
      ctl->tries.waited = 0;
      if (tr.flip) ctl->tries.cur ^= 1;
    }
    ctl->k = k0 + n;
    ctl->timer = timer;
    ctl->nrec = r_hi > ctl->nrec ? r_hi : ctl->nrec;
  }
}

__global__ __launch_bounds__(kFinThreads) void k_finalize(Grid g, Ext ext, Ctl *ctl, int n, const ResGate *gate,
                                                          ResGate *other, int others, ResTry tr) {
  finalize_solve(g, ext, ctl, n, gate, other, others, tr, blockIdx.x == 0);
}

// blockIdx.y = member; a member closes at its scheduled step count.
__global__ __launch_bounds__(kFinThreads) void k_finalize_batch(const SolveDesc *__restrict__ descs, int n,
                                                                const ResGate *gate, ResGate *other, ResTry tr) {
  const SolveDesc &sd = descs[blockIdx.y];
  const bool first = blockIdx.x == 0 && blockIdx.y == 0;
  const int left = sd.nt - sd.d.ctl->k;
  const int n_eff = n < left ? n : left;
  if (gate && first && threadIdx.x == 0) other->arrived = other->decision = 0;
  if (n_eff <= 0) return;
  finalize_solve(sd.g, sd.d.ext, sd.d.ctl, n_eff, gate, other, 0, tr, blockIdx.x == 0);
}

// Whole-field sentinel (no counterpart in the reference, which checks
// nothing): every value of the current fields, as (re, im) pairs, against
// non-finite values and magnitudes above kGrowthLimit; a hit sets status
// bit 1 of the solve.  `!(|x| <= L)` is also true for NaN.  Grid-stride over
// the 2 N M pairs of the state.
__device__ __forceinline__ void sentinel_scan(const double2 *__restrict__ u, size_t n2, Ctl *ctl, size_t i0,
                                              size_t stride) {
  const TEUK_GLOBAL dvec2 *__restrict__ ug = global_ptr(reinterpret_cast<const dvec2 *>(u));
  bool bad = false;
  for (size_t i = i0; i < n2; i += stride) {
    const dvec2 v = ug[i];
    bad = bad || !(fabs(v.x) <= kGrowthLimit) || !(fabs(v.y) <= kGrowthLimit);
  }
  if (bad) atomicOr(&ctl->status, 2);
}

__global__ __launch_bounds__(256) void k_sentinel(const double2 *__restrict__ u, size_t n2, Ctl *ctl) {
  sentinel_scan(u, n2, ctl, (size_t)blockIdx.x * blockDim.x + threadIdx.x, (size_t)gridDim.x * blockDim.x);
}

// blockIdx.y = member; a member that had finished before this chunk (its
// step counter, which the chunk's finalize advances afterwards, is at its
// scheduled count) is skipped.
__global__ __launch_bounds__(256) void k_sentinel_batch(const SolveDesc *__restrict__ descs) {
  const SolveDesc &sd = descs[blockIdx.y];
  if (sd.d.ctl->k >= sd.nt) return;
  const size_t n2 = 2 * (size_t)sd.g.N * sd.g.M;
  sentinel_scan(reinterpret_cast<const double2 *>(sd.d.U), n2, sd.d.ctl,
                (size_t)blockIdx.x * blockDim.x + threadIdx.x, (size_t)gridDim.x * blockDim.x);
}

// ---------------------------------------------------------------------------
// Particle source on the compact ptsx x ptsy patch (kern.cu:770-2683).
#include "teuk_source_dev.inc"

}  // namespace

bool source_available() { return true; }

// ---------------------------------------------------------------------------
// Launchers.
hipError_t launch_init_coeffs(const Grid &g, const DevState &d, hipStream_t s) {
  const size_t NM = (size_t)g.N * g.M;
  const unsigned nb = (unsigned)((NM + 255) / 256);
  hipLaunchKernelGGL(k_init_bb, dim3(nb), dim3(256), 0, s, g, d.ktab, d.rtab, d.scratch);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_init_dbdx, dim3(nb), dim3(256), 0, s, g, d.scratch, d.dbdx);
  return hipGetLastError();
}

static unsigned fields_blocks(size_t NM) { return (unsigned)std::min<size_t>((2 * NM + 255) / 256, 8192); }

hipError_t launch_fields_join(const double *in, double *out, size_t NM, hipStream_t s) {
  hipLaunchKernelGGL(k_fields_join, dim3(fields_blocks(NM)), dim3(256), 0, s, in, out, NM);
  return hipGetLastError();
}

hipError_t launch_fields_split(const double *in, double *out, size_t NM, hipStream_t s) {
  hipLaunchKernelGGL(k_fields_split, dim3(fields_blocks(NM)), dim3(256), 0, s, in, out, NM);
  return hipGetLastError();
}

hipError_t launch_init_res(const Grid &g, const DevState &d, hipStream_t s) {
  hipLaunchKernelGGL(k_init_res, dim3((g.N + 255) / 256), dim3(256), 0, s, g, d);
  return hipGetLastError();
}

hipError_t launch_resident(const Grid &g, const DevState &d, int integrator, bool has_src, ResShape sh,
                           const ResSpan &sp, int nsteps, int nt, ResGate *gate, long long limit, hipStream_t s) {
  if (nsteps < 1 || nsteps > kRing || sp.s0 + (long long)sh.B * sh.C < sp.s1 ||
      sp.s1 - sp.s0 - (long long)(sh.B - 1) * sh.C < 8)
    return hipErrorInvalidValue;
  switch (sh.CP) {
    case 1: return launch_resident_cp<1>(g, d, integrator, has_src, sh, sp, nsteps, nt, gate, limit, s);
    case 2: return launch_resident_cp<2>(g, d, integrator, has_src, sh, sp, nsteps, nt, gate, limit, s);
    case 4: return launch_resident_cp<4>(g, d, integrator, has_src, sh, sp, nsteps, nt, gate, limit, s);
    case 6: return launch_resident_cp<6>(g, d, integrator, has_src, sh, sp, nsteps, nt, gate, limit, s);
    case 8: return launch_resident_cp<8>(g, d, integrator, has_src, sh, sp, nsteps, nt, gate, limit, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_resident_batch(const SolveDesc *descs, const ResBlock *blocks, int nblocks, int integrator, int CP,
                                 int MT, size_t lds, int nsteps, ResGate *gate, long long limit, hipStream_t s) {
  if (nblocks < 1 || nsteps < 1 || nsteps > kRing || lds > kResLdsMax) return hipErrorInvalidValue;
  switch (CP) {
    case 1: return launch_resident_batch_cp<1>(descs, blocks, nblocks, integrator, MT, lds, nsteps, gate, limit, s);
    case 2: return launch_resident_batch_cp<2>(descs, blocks, nblocks, integrator, MT, lds, nsteps, gate, limit, s);
    case 4: return launch_resident_batch_cp<4>(descs, blocks, nblocks, integrator, MT, lds, nsteps, gate, limit, s);
    case 6: return launch_resident_batch_cp<6>(descs, blocks, nblocks, integrator, MT, lds, nsteps, gate, limit, s);
    case 8: return launch_resident_batch_cp<8>(descs, blocks, nblocks, integrator, MT, lds, nsteps, gate, limit, s);
    default: return hipErrorInvalidValue;
  }
}

// Launch shape for an N x M grid, from measurements on an MI355X: 2-row
// wavefronts (2 + (M - 10) / 2 per strip, an odd count, so one wavefront per
// block), compiled for 3 waves per SIMD from M = 64 up; 8-row ones on tall
// grids past the last-level cache; 4-row wavefronts at 8 M points and more, where there are wavefronts enough and fewer theta
// halo re-reads pay.
Tiling default_tiling(int N, int M) {
  Tiling t;
  const bool large = (long long)N * M >= (1LL << 23);
  // Between: the stages no longer live in the last-level cache, and on tall
  // grids 8-row chunks, which re-read the fewest halo rows, win (2-row / 8-row,
  // us a stage: 16000 x 256 SSP-RK3 91.2 / 85.0, RK4 99.6 / 94.7; 24576 x 192
  // 105.2 / 100.0; 8192 x 512 93.2 / 88.7), not on lower ones (32768 x 136 95.0
  // / 99.5) nor below (12288 x 256, 3.1 M points, 59.3 / 61.2).  Above, 4-row
  // chunks (4-row / 8-row, RK4: 32768 x 256 194.0 / 200.4, 45056 x 192 188.0 /
  // 189.3, 65536 x 136 197.4 / 204.3), but for 512 rows and more, which are not
  // told apart here (16384 x 512 207.2 / 196.9, 8192 x 1024 204.2 / 197.6).
  if (!large && (long long)N * M >= 7 * (1LL << 19) && M >= 192) return Tiling{1, 2, 8};
  t.rows = large ? 4 : kDefaultThetaRows;
  t.wpe = (!large && M >= 64) ? 3 : 2;
  const int chunks = theta_chunks(M, t.rows);
  t.wpb = chunks % 4 == 0 ? 4 : (chunks % 2 == 0 ? 2 : 1);
  return t;
}

// Blocks of wpb waves per rho strip; when wpb does not divide the chunks,
// the surplus waves of the last block find no chunk and return at once (the
// stage kernel has no block-level barrier).
int stage_groups(int M, int wpb, int rows) { return (theta_chunks(M, rows) + wpb - 1) / wpb; }

hipError_t launch_stage(const Grid &g, const DevState &d, int integrator, int stage, bool has_src, int k_rel,
                        Tiling t, hipStream_t s) {
  if (t.wpb < 1 || t.wpb > 4 || !theta_rows_ok(g.M, t.rows)) return hipErrorInvalidValue;
  const int ngroups = stage_groups(g.M, t.wpb, t.rows);
  const int nb = (g.N / kWave) * ngroups;
  const dim3 grid(nb), block(kWave, t.wpb);
  switch (t.rows) {
    case 2: return launch_stage_rows<2>(g, d, integrator, stage, has_src, k_rel, ngroups, grid, block, t.wpe, s);
    case 4: return launch_stage_rows<4>(g, d, integrator, stage, has_src, k_rel, ngroups, grid, block, t.wpe, s);
    case 8: return launch_stage_rows<8>(g, d, integrator, stage, has_src, k_rel, ngroups, grid, block, t.wpe, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_stage_batch(const BatchTile *tiles, int ntiles, int integrator, int stage, int k_rel, Tiling t,
                              hipStream_t s) {
  if (ntiles <= 0) return hipSuccess;
  if (t.wpb < 1 || t.wpb > 4) return hipErrorInvalidValue;
  const dim3 block(kWave, t.wpb);
  switch (t.rows) {
    case 2: return launch_stage_batch_rows<2>(tiles, ntiles, integrator, stage, k_rel, block, t.wpe, s);
    case 4: return launch_stage_batch_rows<4>(tiles, ntiles, integrator, stage, k_rel, block, t.wpe, s);
    case 8: return launch_stage_batch_rows<8>(tiles, ntiles, integrator, stage, k_rel, block, t.wpe, s);
    default: return hipErrorInvalidValue;
  }
}

// A block for each record that n steps can hold (at least one block).
static unsigned finalize_blocks(int n, int Fr) {
  const int most = (std::max(n, 1) - 1) / std::max(Fr, 1) + 1;
  return (unsigned)std::min(most, 2 * kRing);
}

hipError_t launch_finalize_batch(const SolveDesc *descs, int nsolves, int n, ResGate *gate, ResGate *other, ResTry t,
                                 hipStream_t s) {
  if (nsolves <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_finalize_batch, dim3(finalize_blocks(n, 1), nsolves), dim3(kFinThreads), 0, s, descs, n, gate,
                     other, t);
  return hipGetLastError();
}

hipError_t launch_source_batch(const SolveDesc *descs, int nsolves, int max_cells, int k_rel0, int n,
                               bool colmajor, hipStream_t s) {
  if (nsolves <= 0 || max_cells <= 0 || n <= 0) return hipSuccess;
  if (n > kRing) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_source_batch, dim3((max_cells + 255) / 256, nsolves, n), dim3(256), 0, s, descs, k_rel0,
                     colmajor);
  return hipGetLastError();
}

hipError_t launch_finalize(const Grid &g, const DevState &d, int n, ResGate *gate, ResGate *other, ResTry t,
                           hipStream_t s, int others) {
  hipLaunchKernelGGL(k_finalize, dim3(finalize_blocks(n, g.Fr)), dim3(kFinThreads), 0, s, g, d.ext, d.ctl, n, gate,
                     other, others, t);
  return hipGetLastError();
}

// Blocks of 256 threads, about four pairs per thread, at most 1024 blocks.
static unsigned sentinel_blocks(size_t n2) {
  const size_t nb = (n2 + 1023) / 1024;
  return (unsigned)(nb < 1 ? 1 : (nb > 1024 ? 1024 : nb));
}

hipError_t launch_sentinel(const Grid &g, const DevState &d, hipStream_t s) {
  const size_t n2 = 2 * (size_t)g.N * g.M;
  hipLaunchKernelGGL(k_sentinel, dim3(sentinel_blocks(n2)), dim3(256), 0, s,
                     reinterpret_cast<const double2 *>(d.U), n2, d.ctl);
  return hipGetLastError();
}

hipError_t launch_sentinel_batch(const SolveDesc *descs, int nsolves, hipStream_t s) {
  if (nsolves <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sentinel_batch, dim3(64, nsolves), dim3(256), 0, s, descs);
  return hipGetLastError();
}

hipError_t launch_source(const Grid &g, const DevState &d, int k_rel0, int n, bool colmajor, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (n > kRing) return hipErrorInvalidValue;
  const int cells = g.ptsx * g.ptsy;
  hipLaunchKernelGGL(k_source, dim3((cells + 255) / 256, n), dim3(256), 0, s, g, d, k_rel0, colmajor);
  return hipGetLastError();
}

hipError_t launch_source_at(const Grid &g, const DevState &d, int kstep, hipStream_t s) {
  const int cells = g.ptsx * g.ptsy;
  hipLaunchKernelGGL(k_source_at, dim3((cells + 255) / 256), dim3(256), 0, s, g, d, kstep);
  return hipGetLastError();
}

hipError_t launch_source_coeffs(const teuk_t4::StepIn *in, SrcDev *sched, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_source_coeffs, dim3((n + 63) / 64), dim3(64), 0, s, in, sched, n);
  return hipGetLastError();
}

}  // namespace teuk
