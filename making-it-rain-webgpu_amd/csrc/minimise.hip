// minimise.hip -- the device side of md_minimise: the L-BFGS vectors, the
// OpenMM objective's gradient with constraint springs, and the reductions
// the search reads back as scalars.
//
// Replaces the upload / evaluate / read-back loop of upstream's
// minimiseOnDevice (src/gpu/minimise.ts:33-54), whose L-BFGS runs on the
// host (src/reference/minimise.ts:164-280, lbfgs.ts:102-275): here every
// 3N-vector -- positions, gradient, direction, trial point, the six
// correction pairs -- stays in HBM as f64 planes [3][np], and the host only
// reads back the few scalars the line search decides on, once per trial point
// and once per search direction.  Reductions run in a fixed order (per-block
// partial sums, then those in block order), so a minimisation is reproducible
// run to run.
//
// At the sizes a minimisation is run at (9k atoms: 27k components) every kernel
// here is a few us of latency, so what counts is how many there are and how
// often the host waits.  Finishing each dot product in a kernel of its own and
// waiting for it cost 14 round trips a direction and three a trial: of 590 us
// an evaluation of the objective, some 335 us.  Now a reduction is finished by
// the kernel that needs it (every block adds the same partials in the same
// order), the two-loop recursion takes one launch per correction vector with
// its coefficients kept on the device, and a trial point's values come back
// together.  Ten iterations a round at 9k atoms, 98 evaluations: 57.7 ms before,
// 29.3 so (and 21.2 with what the evaluation has gained since).
#include "engine.hpp"

#define MD_MIN_BLOCK 256
#define MD_MIN_PARTIALS 1024  // most blocks a reduction uses (then grid-strided)

static int blocks_for(int count) { return std::max(1, std::min(MD_MIN_PARTIALS, (count + MD_MIN_BLOCK - 1) / MD_MIN_BLOCK)); }

__device__ __forceinline__ double md_block_sum(double v) {
  __shared__ double part[MD_MIN_BLOCK / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < MD_MIN_BLOCK / 64; ++w) s += part[w];
  __syncthreads();
  return s;
}

__device__ __forceinline__ double md_block_max(double v) {
  __shared__ double part[MD_MIN_BLOCK / 64];
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < MD_MIN_BLOCK / 64; ++w) s = fmax(s, part[w]);
  __syncthreads();
  return s;
}

// partial[0 .. count) added in order (or its maximum), in every thread of the
// block; `part` is LDS for MD_MIN_PARTIALS values.
template <bool MAX>
__device__ __forceinline__ double md_min_finish(const double *partial, int count, double *part) {
  __syncthreads();  // `part` may hold an earlier reduction's values still being read
  for (int b = threadIdx.x; b < count; b += blockDim.x) part[b] = partial[b];
  __syncthreads();
  double s = 0.0;
#pragma unroll 8
  for (int b = 0; b < count; ++b) s = MAX ? fmax(s, part[b]) : s + part[b];
  return s;
}

// ---- vector kernels over the 3 planes of n real atoms (pitch np) -------------
//
// The sums and products below round as a * x + (b y) and a * b + s do: the
// second product of a combination is rounded, the first is fused (__builtin_fma
// says so, not the compiler's choice).

// partial[0 .. count) -> *out in order (sum or max), through LDS so that the
// loads are in flight together
__global__ void k_min_finish(const double *partial, int count, int max, double *out) {
  __shared__ double part[MD_MIN_PARTIALS];
  const double v = max ? md_min_finish<true>(partial, count, part) : md_min_finish<false>(partial, count, part);
  if (threadIdx.x == 0) *out = v;
}

// Q32.32 positions <-> f64 nm
__global__ void k_min_from_fixed(const int64_t *pos, double *x, int n, int np) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < 3 * n; k += gridDim.x * blockDim.x) {
    const int d = k / n, i = k - d * n;
    x[d * np + i] = md_fixed_to_double_dev(pos[d * np + i]);
  }
}

// positions from x (rounded to Q32.32 as md_set_positions rounds); the drift
// residual cleared; *bad set when a coordinate is outside +/-2^31 nm.  Given a
// direction d the positions are trial = x + step d.  The control block is set
// as the host sets it before an evaluation: the list rebuilt, the step counter.
__global__ void k_min_to_fixed(const double *x, const double *d, double step, double *trial, int64_t *pos, float *resid,
                               int n, int np, int *bad, md_control *ctl, int64_t steps) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < 3 * n; k += gridDim.x * blockDim.x) {
    const int p = k / n, at = p * np + (k - p * n);
    double v = x[at];
    if (d) {
      v = __builtin_fma(1.0, v, step * d[at]);
      trial[at] = v;
    }
    if (!(fabs(v) < 2147483648.0)) {
      *bad = 1;
      continue;
    }
    pos[at] = (int64_t)rint(v * 4294967296.0);
    resid[at] = 0.0f;
  }
  if (ctl && blockIdx.x == 0 && threadIdx.x == 0) {
    ctl->overflow = 0;
    ctl->force_pending = 1;
    ctl->step_next = steps;
  }
}

// One constraint spring of OpenMM's minimiser objective, (k/2)(r - d)^2: the
// separation of its atoms and the pull per unit of it.
__device__ __forceinline__ double md_min_spring(const double *x, int np, int a, int b, double dist, double kspring,
                                                double v[3], double &dr) {
  for (int d = 0; d < 3; ++d) v[d] = x[d * np + a] - x[d * np + b];
  const double r2 = __builtin_fma(v[2], v[2], __builtin_fma(v[0], v[0], v[1] * v[1]));
  const double r = sqrt(r2);
  dr = r - dist;
  return kspring * dr / (r == 0.0 ? 1.0 : r);
}

// The objective's gradient at x: -F for moving atoms plus their springs' pulls
// in the order of the atom's list (each spring found again by both its atoms, a
// component each: no pass that stores pulls, no atomics), 0 for frozen ones.
// Its products with the direction and with itself and the springs' energy go
// into partials 0, 1 and 2.
__global__ void __launch_bounds__(MD_MIN_BLOCK)
    k_min_gradient(const int64_t *force, const float *inv_mass, const double *x, const double *dir, const int *p1,
                   const int *p2, const double *dist, int nc, double kspring, const int *cstart, const int *clist,
                   double *g, int n, int np, int blocks, int spring_blocks, double *partial) {
  if ((int)blockIdx.x < blocks) {
    double slope = 0.0, gg = 0.0;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < 3 * n; k += blocks * blockDim.x) {
#pragma clang fp contract(off)
      const int p = k / n, i = k - p * n;
      const int at = p * np + i;
      double v = 0.0;
      if (inv_mass[i] != 0.0f) {
        v = -md_fixed_to_double_dev(force[at]);
        const int first = nc ? cstart[i] : 0, end = nc ? cstart[i + 1] : 0;
        if (first != end) {
          double sum = 0.0;
          for (int c = first; c < end; ++c) {
            const int code = clist[c], spring = code >= 0 ? code : -code - 1;
            double sep[3], dr;
            const double f = md_min_spring(x, np, p1[spring], p2[spring], dist[spring], kspring, sep, dr);
            const double pull = f * (p == 0 ? sep[0] : p == 1 ? sep[1] : sep[2]);
            sum += code >= 0 ? pull : -pull;
          }
          v += sum;
        }
      }
      g[at] = v;
      if (dir) slope = __builtin_fma(v, dir[at], slope);
      gg = __builtin_fma(v, v, gg);
    }
    slope = md_block_sum(slope);
    gg = md_block_sum(gg);
    if (threadIdx.x == 0) {
      partial[blockIdx.x] = slope;
      partial[MD_MIN_PARTIALS + blockIdx.x] = gg;
    }
  }
  if ((int)blockIdx.x < spring_blocks) {
    double e = 0.0;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nc; c += spring_blocks * blockDim.x) {
      double sep[3], dr;
      md_min_spring(x, np, p1[c], p2[c], dist[c], kspring, sep, dr);
      e = __builtin_fma(dr, 0.5 * kspring * dr, e);
    }
    e = md_block_sum(e);
    if (threadIdx.x == 0) partial[2 * MD_MIN_PARTIALS + blockIdx.x] = e;
  }
}

// d = -g, with g.d and the largest |d| into partials 6 and 7
__global__ void k_min_steepest(const double *g, double *d, int n, int np, double *partial) {
  double slope = 0.0, most = 0.0;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < 3 * n; k += gridDim.x * blockDim.x) {
    const int p = k / n, at = p * np + (k - p * n);
    const double v = 0.0 - g[at];
    d[at] = v;
    slope = __builtin_fma(g[at], v, slope);
    most = fmax(most, fabs(v));
  }
  slope = md_block_sum(slope);
  most = md_block_max(most);
  if (threadIdx.x == 0) {
    partial[6 * MD_MIN_PARTIALS + blockIdx.x] = slope;
    partial[7 * MD_MIN_PARTIALS + blockIdx.x] = most;
  }
}

// ---- the two-loop recursion: q = -H g --------------------------------------------
//
// One launch forms the step's correction pair, then one per vector update: each
// finishes the dot product its coefficient needs from the partials of the launch
// before and leaves the next one's.  Whether the pair is kept (S.Y > 0) is
// decided on the device; the host launches for the most pairs there can be, and
// a launch past the count does nothing.  Partials 4 and 5 alternate, so no block
// reads what another of the same launch writes.

// Pairs held once this step's is judged, and the slot of the k-th newest.
__device__ __forceinline__ int md_min_held(const md_min_loop &L, int kept) {
  return kept ? min(L.count + 1, MD_MIN_MEMORY) : L.count;
}
__device__ __forceinline__ int md_min_slot(const md_min_loop &L, int kept, int k) {
  return (L.head + (kept ? 1 : 0) - 1 - k + 2 * MD_MIN_MEMORY) % MD_MIN_MEMORY;
}

// The pair S = trial - x, Y = gt - g into slot head; q = -gt; S.Y, Y.Y, S.q and
// the newest older pair's S.q into partials 0 to 3.
__global__ void __launch_bounds__(MD_MIN_BLOCK)
    k_min_pair(md_min_loop L, const double *x, const double *trial, const double *g) {
  double *S = L.S[L.head], *Y = L.Y[L.head];
  const double *older = L.count ? L.S[(L.head - 1 + MD_MIN_MEMORY) % MD_MIN_MEMORY] : nullptr;
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < 3 * L.n; k += gridDim.x * blockDim.x) {
    const int p = k / L.n, at = p * L.np + (k - p * L.n);
    const double s = trial[at] - x[at], y = L.g[at] - g[at], v = 0.0 - L.g[at];
    S[at] = s;
    Y[at] = y;
    L.q[at] = v;
    sum[0] = __builtin_fma(s, y, sum[0]);
    sum[1] = __builtin_fma(y, y, sum[1]);
    sum[2] = __builtin_fma(s, v, sum[2]);
    if (older) sum[3] = __builtin_fma(older[at], v, sum[3]);
  }
  for (int j = 0; j < 4; ++j) {
    sum[j] = md_block_sum(sum[j]);
    if (threadIdx.x == 0) L.partial[j * MD_MIN_PARTIALS + blockIdx.x] = sum[j];
  }
}

// The k-th step of the first loop (newest to oldest; BACK: of the second, back
// to the newest).
template <bool BACK>
__global__ void __launch_bounds__(MD_MIN_BLOCK) k_min_loop(md_min_loop L, int k) {
#pragma clang fp contract(off)
  __shared__ double part[MD_MIN_PARTIALS];
  const int blocks = gridDim.x;
  const bool first = !BACK && k == 0;
  double sy = 0.0, yy = 0.0;
  int kept;
  if (first) {
    sy = md_min_finish<false>(L.partial, blocks, part);
    yy = md_min_finish<false>(L.partial + MD_MIN_PARTIALS, blocks, part);
    kept = sy > 0.0;
  } else {
    kept = L.state->kept;
  }
  const int held = md_min_held(L, kept);
  if (k >= held && !first) return;
  double *from = L.partial + (4 + (k & 1)) * MD_MIN_PARTIALS, *to = L.partial + (4 + (k & 1)) * MD_MIN_PARTIALS;
  if (first) from = L.partial + (kept ? 2 : 3) * MD_MIN_PARTIALS;
  else if (!BACK) from = L.partial + (4 + ((k - 1) & 1)) * MD_MIN_PARTIALS;
  else to = L.partial + (4 + ((k - 1) & 1)) * MD_MIN_PARTIALS;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (first && lead) {
    L.state->kept = kept;
    if (kept) {
      L.state->rho[L.head] = 1.0 / sy;
      L.state->yy[L.head] = yy;
    }
  }
  const int slot = md_min_slot(L, kept, k);
  const bool last = !BACK && k == held - 1, end = BACK ? k == 0 : held == 0;
  double c = 0.0, scale = 1.0;
  const double *add = BACK ? L.S[slot] : L.Y[slot], *next;
  if (held) {
    const int newest = md_min_slot(L, kept, 0);
    const double rho = first && kept ? 1.0 / sy : L.state->rho[slot];
    const double dot = md_min_finish<false>(from, blocks, part);
    if (BACK) {
      c = L.state->alpha[k] - rho * dot;
    } else {
      const double alpha = rho * dot;
      c = -alpha;
      if (lead) L.state->alpha[k] = alpha;
      if (last) {
        const double rho0 = first ? rho : L.state->rho[newest];
        scale = 1.0 / (rho0 * (first && kept ? yy : L.state->yy[newest]));
      }
    }
  }
  next = end ? L.g : BACK ? L.Y[md_min_slot(L, kept, k - 1)] : last ? L.Y[slot] : L.S[md_min_slot(L, kept, k + 1)];
  double sum = 0.0, most = 0.0;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < 3 * L.n; e += gridDim.x * blockDim.x) {
    const int p = e / L.n, at = p * L.np + (e - p * L.n);
    double v = L.q[at];
    if (held) {
      v = v + c * add[at];
      if (last) v = __builtin_fma(scale, v, 0.0);
      L.q[at] = v;
    }
    sum = __builtin_fma(next[at], v, sum);
    most = fmax(most, fabs(v));
  }
  sum = md_block_sum(sum);
  most = md_block_max(most);
  if (threadIdx.x == 0) {
    if (end) {
      L.partial[6 * MD_MIN_PARTIALS + blockIdx.x] = sum;
      L.partial[7 * MD_MIN_PARTIALS + blockIdx.x] = most;
    } else {
      to[blockIdx.x] = sum;
    }
  }
}

// ---- what the host reads: one workgroup into pinned memory ------------------------

// a trial point: its energies, the errors it raised, and the sums k_min_gradient left
__global__ void __launch_bounds__(MD_MIN_BLOCK)
    k_min_report_trial(const double *partial, int blocks, int spring_blocks, int *bad, const md_control *ctl,
                       const int64_t *energy, md_min_report *out) {
  __shared__ double part[MD_MIN_PARTIALS];
  const double slope = md_min_finish<false>(partial, blocks, part);
  const double gg = md_min_finish<false>(partial + MD_MIN_PARTIALS, blocks, part);
  const double spring = md_min_finish<false>(partial + 2 * MD_MIN_PARTIALS, spring_blocks, part);
  for (int k = threadIdx.x; k < MD_E_SLOTS; k += blockDim.x) out->energy[k] = energy[k];
  if (threadIdx.x == 0) {
    out->slope = slope;
    out->gg = gg;
    out->spring = spring;
    out->bad = *bad;
    out->errors = {ctl->step_current, ctl->overflow, ctl->barostat_error, ctl->diverged};
    *bad = 0;
  }
}

// a direction: its slope and largest component, and whether the pair was kept
__global__ void __launch_bounds__(MD_MIN_BLOCK)
    k_min_report_direction(const double *partial, int blocks, const md_min_state *state, md_min_report *out) {
  __shared__ double part[MD_MIN_PARTIALS];
  const double slope = md_min_finish<false>(partial + 6 * MD_MIN_PARTIALS, blocks, part);
  const double most = md_min_finish<true>(partial + 7 * MD_MIN_PARTIALS, blocks, part);
  if (threadIdx.x == 0) {
    out->slope = slope;
    out->most = most;
    out->kept = state->kept;
  }
}

// the largest relative constraint deviation |r - d| / d, per block
__global__ void k_min_constraint_error(const double *x, const int *p1, const int *p2, const double *dist, int nc,
                                       int np, double *partial) {
  double w = 0.0;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nc; c += gridDim.x * blockDim.x) {
    const int a = p1[c], b = p2[c];
    double r2 = 0.0;
    for (int d = 0; d < 3; ++d) {
      const double v = x[d * np + a] - x[d * np + b];
      r2 += v * v;
    }
    w = fmax(w, fabs(sqrt(r2) - dist[c]) / dist[c]);
  }
  w = md_block_max(w);
  if (threadIdx.x == 0) partial[blockIdx.x] = w;
}

// ---- host launchers (engine.hpp) ---------------------------------------------

md_min_work *md_min_work_create(md_system *s, const std::vector<int> &p1, const std::vector<int> &p2,
                                const std::vector<double> &dist) {
  std::unique_ptr<md_min_work> w(new md_min_work());
  MD_HIP(hipHostMalloc(&w->report, sizeof(md_min_report)));
  const size_t len = 3 * (size_t)s->np;
  w->vec = md_alloc<double>(s, len * MD_MIN_VECTORS);
  w->partial = md_alloc<double>(s, 8 * MD_MIN_PARTIALS);
  w->state = md_alloc<md_min_state>(s, 1);
  w->scalar = md_alloc<double>(s, 1);
  w->bad = md_alloc<int>(s, 1);
  w->nc = (int)p1.size();
  w->p1 = md_alloc<int>(s, std::max<size_t>(1, p1.size()));
  w->p2 = md_alloc<int>(s, std::max<size_t>(1, p2.size()));
  w->dist = md_alloc<double>(s, std::max<size_t>(1, dist.size()));
  // by atom, the springs that pull it (first atoms +c, second atoms -c - 1)
  std::vector<int> cstart(s->np + 1, 0), clist(2 * p1.size());
  for (size_t c = 0; c < p1.size(); ++c) {
    ++cstart[p1[c] + 1];
    ++cstart[p2[c] + 1];
  }
  for (int a = 0; a < s->np; ++a) cstart[a + 1] += cstart[a];
  {
    std::vector<int> fill(cstart.begin(), cstart.end() - 1);
    for (size_t c = 0; c < p1.size(); ++c) {
      clist[fill[p1[c]]++] = (int)c;
      clist[fill[p2[c]]++] = -(int)c - 1;
    }
  }
  w->cstart = md_alloc<int>(s, cstart.size());
  w->clist = md_alloc<int>(s, std::max<size_t>(1, clist.size()));
  MD_HIP(hipMemcpyAsync(w->cstart, cstart.data(), sizeof(int) * cstart.size(), hipMemcpyHostToDevice, s->stream));
  if (!clist.empty())
    MD_HIP(hipMemcpyAsync(w->clist, clist.data(), sizeof(int) * clist.size(), hipMemcpyHostToDevice, s->stream));
  if (w->nc) {
    MD_HIP(hipMemcpyAsync(w->p1, p1.data(), sizeof(int) * p1.size(), hipMemcpyHostToDevice, s->stream));
    MD_HIP(hipMemcpyAsync(w->p2, p2.data(), sizeof(int) * p2.size(), hipMemcpyHostToDevice, s->stream));
    MD_HIP(hipMemcpyAsync(w->dist, dist.data(), sizeof(double) * dist.size(), hipMemcpyHostToDevice, s->stream));
  }
  MD_HIP(hipStreamSynchronize(s->stream));
  return w.release();
}

double *md_min_vec(md_system *s, md_min_work *w, int k) { return w->vec + (size_t)k * 3 * s->np; }

static double read_scalar(md_system *s, md_min_work *w) {
  double v = 0.0;
  MD_HIP(hipMemcpyAsync(&v, w->scalar, sizeof v, hipMemcpyDeviceToHost, s->stream));
  MD_HIP(hipStreamSynchronize(s->stream));
  return v;
}

void md_min_positions_out(md_system *s, double *x) {
  k_min_from_fixed<<<blocks_for(3 * s->n), MD_MIN_BLOCK, 0, s->stream>>>(s->pos, x, s->n, s->np);
  MD_HIP(hipGetLastError());
}

bool md_min_positions_in(md_system *s, md_min_work *w, const double *x) {
  MD_HIP(hipMemsetAsync(w->bad, 0, sizeof(int), s->stream));
  k_min_to_fixed<<<blocks_for(3 * s->n), MD_MIN_BLOCK, 0, s->stream>>>(x, nullptr, 0.0, nullptr, s->pos, s->resid, s->n,
                                                                      s->np, w->bad, nullptr, 0);
  MD_HIP(hipGetLastError());
  int bad = 0;
  MD_HIP(hipMemcpyAsync(&bad, w->bad, sizeof bad, hipMemcpyDeviceToHost, s->stream));
  MD_HIP(hipStreamSynchronize(s->stream));
  return bad == 0;
}

void md_min_trial(md_system *s, md_min_work *w, const double *x, const double *d, double step, double *trial) {
  k_min_to_fixed<<<blocks_for(3 * s->n), MD_MIN_BLOCK, 0, s->stream>>>(x, d, step, trial, s->pos, s->resid, s->n, s->np,
                                                                      w->bad, s->ctl, s->steps_done);
  MD_HIP(hipGetLastError());
}

const md_min_report &md_min_gradient(md_system *s, md_min_work *w, const double *x, const double *d, double kspring,
                                     double *g) {
  const int blocks = blocks_for(3 * s->n), spring_blocks = w->nc ? blocks_for(w->nc) : 0;
  k_min_gradient<<<std::max(blocks, spring_blocks), MD_MIN_BLOCK, 0, s->stream>>>(
      s->force, s->inv_mass, x, d, w->p1, w->p2, w->dist, w->nc, kspring, w->cstart, w->clist, g, s->n, s->np, blocks,
      spring_blocks, w->partial);
  k_min_report_trial<<<1, MD_MIN_BLOCK, 0, s->stream>>>(w->partial, blocks, spring_blocks, w->bad, s->ctl, s->energy,
                                                       w->report);
  MD_HIP(hipGetLastError());
  MD_HIP(hipStreamSynchronize(s->stream));
  return *w->report;
}

static const md_min_report &read_direction(md_system *s, md_min_work *w) {
  k_min_report_direction<<<1, MD_MIN_BLOCK, 0, s->stream>>>(w->partial, blocks_for(3 * s->n), w->state, w->report);
  MD_HIP(hipGetLastError());
  MD_HIP(hipStreamSynchronize(s->stream));
  return *w->report;
}

const md_min_report &md_min_steepest(md_system *s, md_min_work *w, const double *g, double *d) {
  k_min_steepest<<<blocks_for(3 * s->n), MD_MIN_BLOCK, 0, s->stream>>>(g, d, s->n, s->np, w->partial);
  return read_direction(s, w);
}

const md_min_report &md_min_direction(md_system *s, md_min_work *w, md_min_loop L, const double *x,
                                      const double *trial, const double *g) {
  const int blocks = blocks_for(3 * s->n), most = std::min(L.count + 1, MD_MIN_MEMORY);
  L.n = s->n;
  L.np = s->np;
  L.partial = w->partial;
  L.state = w->state;
  k_min_pair<<<blocks, MD_MIN_BLOCK, 0, s->stream>>>(L, x, trial, g);
  for (int k = 0; k < most; ++k) k_min_loop<false><<<blocks, MD_MIN_BLOCK, 0, s->stream>>>(L, k);
  for (int k = most - 1; k >= 0; --k) k_min_loop<true><<<blocks, MD_MIN_BLOCK, 0, s->stream>>>(L, k);
  return read_direction(s, w);
}

double md_min_constraint_error(md_system *s, md_min_work *w, const double *x) {
  if (!w->nc) return 0.0;
  const int nb = blocks_for(w->nc);
  k_min_constraint_error<<<nb, MD_MIN_BLOCK, 0, s->stream>>>(x, w->p1, w->p2, w->dist, w->nc, s->np, w->partial);
  k_min_finish<<<1, MD_MIN_BLOCK, 0, s->stream>>>(w->partial, nb, 1, w->scalar);
  MD_HIP(hipGetLastError());
  return read_scalar(s, w);
}
