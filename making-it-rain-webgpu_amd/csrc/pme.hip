// pme.hip -- smooth particle-mesh Ewald for gfx950.
//
// Replaces the upstream WGSL `spread_charge` (src/gpu/kernels/pme.wgsl:123-154),
// `load_grid` (pme-grid.wgsl:13-19), `fft_stage` (fft.wgsl:59-107), `convolve`
// (pme-convolve.wgsl:33-91) and `interpolate_force` (pme-interpolate.wgsl
// :104-155).  The mathematics is src/reference/forces/pme.ts:94-263: order-5
// cardinal B-splines at fractional coordinates (grid points floor(u)-4 ..
// floor(u)), E = (2 pi K / V) sum_{m != 0} exp(-k^2/4 alpha^2) / (k^2 |b(m)|^2)
// |Q(m)|^2 with k = 2 pi m B^-T, the grid multiplied by twice the factor, and
// forces -q B^-1 (n_x dtheta_x theta_y theta_z, ...) . phi.
//
// gfx950 design: the charge grid is int64 Q32.32 (125 atomic adds per charged
// atom, order independent); the transform is real-to-complex, so only
// nz/2+1 planes of k-space are stored and transformed; each 1D transform runs
// whole inside LDS (a batch of lines per workgroup, mixed-radix Stockham
// stages, twiddles from an f64-computed table); the x-axis pass does forward
// transform, convolution, energy and inverse transform in one kernel; the
// z pass that reads the integer grid also clears it for the next step.
#include <climits>
#include <cmath>
#include <vector>

#include "engine.hpp"

#define PME_MAX_STAGES 12
#define PME_BATCH 16          // lines of a workgroup, at most (md_lines)
#define PME_LDS (160 * 1024)  // a CU's LDS
#define MD_PHI_PAD 4  // values a row of the potential repeats past its end (md_row5)

struct md_fft_plan {
  int n;
  int nstages;
  int radix[PME_MAX_STAGES];
  int tw;  // offset of this length's twiddle table
  int lines;      // lines of a workgroup
  int runs, per;  // for lines along y or x: a row's runs of consecutive kz, and the kz of a run
};

struct md_pme_args {
  int nx, ny, nz, nzc;
  md_fft_plan px, py, pz;
  const float2 *tw;  // exp(-2 pi i t / n), per length
  const float *mod_x, *mod_y, *mod_z;
  double inv[9];
  float invf[9];
  float prefactor;   // K 2 pi / V
  float exp_scale;   // -1/(4 alpha^2)
};

// one replica's table entry
struct md_pme_table {
  md_pme_args P;
  int n, np, nslots;
  const int64_t *pos;
  const float4 *param;
  const int *slot_atom;  // the nonbonded list's spatial order, 64-slot super-clusters
  int64_t *grid;
  float2 *cgrid;
  float *phi;
  int64_t *force;
  int64_t *energy;
  int small_charges;  // every |charge| < MD_SMALL_FIXED
  md_pair_forces F;
  const int64_t *piece;  // the bonded terms' pieces, by atom
  const int *piece_start;
};

__device__ __forceinline__ const md_pme_table &md_pme_entry(const md_pme_table *T, const md_bmap &map, int &blk) {
  return T[md_locate(map, blockIdx.x, blk)];
}

// ---- B-splines (src/reference/forces/bspline.ts:55-91, order 5) ------------

__device__ __forceinline__ void md_bspline5(float w, float *th, float *dth) {
  float l0 = 1.0f - w, l1 = w, l2, l3;
  // order 3
  l2 = 0.5f * w * l1;
  l1 = 0.5f * ((w + 1.0f) * l0 + (2.0f - w) * l1);
  l0 = 0.5f * (1.0f - w) * l0;
  // order 4
  const float third = 1.0f / 3.0f;
  l3 = third * w * l2;
  l2 = third * ((w + 1.0f) * l1 + (3.0f - w) * l2);
  l1 = third * ((w + 2.0f) * l0 + (2.0f - w) * l1);
  l0 = third * (1.0f - w) * l0;
  if (dth) {
    dth[0] = -l0;
    dth[1] = l0 - l1;
    dth[2] = l1 - l2;
    dth[3] = l2 - l3;
    dth[4] = l3;
  }
  // order 5
  th[4] = 0.25f * w * l3;
  th[3] = 0.25f * ((w + 1.0f) * l2 + (4.0f - w) * l3);
  th[2] = 0.25f * ((w + 2.0f) * l1 + (3.0f - w) * l2);
  th[1] = 0.25f * ((w + 3.0f) * l0 + (2.0f - w) * l1);
  th[0] = 0.25f * (1.0f - w) * l0;
}

// fractional position on the mesh, from the exact fixed-point coordinate
__device__ __forceinline__ void md_mesh_coord(const int64_t *pos, int np, int i, const double *M, int nx, int ny,
                                              int nz, int *base, float *w) {
  const double s = 2.3283064365386963e-10;
  double rx = (double)pos[i] * s, ry = (double)pos[np + i] * s, rz = (double)pos[2 * np + i] * s;
  double f[3] = {rx * M[0] + ry * M[3] + rz * M[6], ry * M[4] + rz * M[7], rz * M[8]};
  int n[3] = {nx, ny, nz};
  for (int d = 0; d < 3; ++d) {
    double fr = f[d] - floor(f[d]);
    double u = fr * n[d];
    double cell = floor(u);
    w[d] = (float)(u - cell);
    base[d] = (int)cell - (MD_PME_ORDER - 1);
  }
}

__device__ __forceinline__ int md_wrap(int i, int n) {
  i %= n;
  return i < 0 ? i + n : i;
}

// a stencil point's mesh index: from -4 (a base is a cell minus 4) to n, and n
// is at least the spline's order
__device__ __forceinline__ int md_wrap_once(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// md_to_fixed for |x| < 2^19: adding 1.5 * 2^20 in f64 rounds x to a multiple of
// 2^-32, ties to even, and leaves that multiple in the sum's low bits.  Four
// instructions instead of about twelve.
__device__ __forceinline__ int64_t md_small_to_fixed(float x) {
  return __double_as_longlong((double)x + 1572864.0) - 0x4138000000000000ll;
}
#define MD_SMALL_FIXED 524288.0f  // 2^19

// idx / m for 0 <= idx < 2^20 by an f32 reciprocal (an integer division is some
// 30 instructions, more than a radix-4 butterfly): (idx + 1/2) / m is at least
// 1/(2m) from an integer, and the product is within 3.6e-7 of it relatively.
__device__ __forceinline__ float md_inverse(int m) { return __builtin_amdgcn_rcpf((float)m); }
__device__ __forceinline__ int md_div(int idx, float inv) { return (int)(((float)idx + 0.5f) * inv); }

// the representative in [-n/2, n/2) of a difference of two bases
__device__ __forceinline__ int md_wrap_near(int d, int n) {
  if (d < 0) d += n;  // bases lie in [-4, n]: now in [0, n + 4]
  if (d >= n) d -= n;
  return d >= n / 2 ? d - n : d;
}

// Charge spreading.  A workgroup takes `per` consecutive 64-slot super-clusters
// of the nonbonded list (spatially compact: their atoms' stencils overlap); one
// wave each finds the atoms' stencils, then wave a adds plane a of every stencil
// to an int64 tile in LDS covering their stencil box, and the tile is added to
// the grid, one global atomic per non-zero point: about a fifth of the atomics
// of spreading atom by atom.  Contributions are Q32.32 and integer sums do not
// depend on order, so the grid is the same however atoms are grouped.  Super-
// clusters whose joint box exceeds the tile go one at a time; a single one that
// exceeds it spreads straight to the grid.
//
// Bound by the atomic requests at memory, and on small launches by latency (64
// replicas, 289 us before, with 4.6 M requests and 91 M wave instructions, 150
// us of VALU issue): stencils are found once, not by each of the five waves,
// contributions are rounded by md_small_to_fixed, the flush divides by
// reciprocals, and two super-clusters share a tile where there are enough of
// them to fill the chip.  Now 258 us there, 85 at 243k atoms (107), 15 at 31k
// (18).
#define MD_SPREAD_WAVES MD_PME_ORDER
#define MD_SPREAD_THREADS (64 * MD_SPREAD_WAVES)
#define MD_SPREAD_TILE 5632  // int64 points: 45 KB, with the stencils 54 KB, three workgroups to a CU
#define MD_SPREAD_MOST 2     // super-clusters of a workgroup
#define MD_SPREAD_PAIRED 1024  // super-clusters of a launch from which they go two to a workgroup

struct md_spread_box {
  int ref[3], lo[3], hi[3];  // a stencil base, and the lowest and highest offsets from it; lo > hi: no charge
};

__global__ void __launch_bounds__(MD_SPREAD_THREADS) k_pme_spread(const md_pme_table *__restrict__ T, md_bmap map, int per) {
  // super-clusters laid out XCD by XCD: neighbouring ones add into the same
  // mesh region from one L2
  int blk;
  const md_pme_table &E = T[md_locate(map, md_xcd_block(blockIdx.x, gridDim.x), blk)];
  const md_pme_args &P = E.P;
  int64_t *grid = E.grid;
  __shared__ unsigned long long tile[MD_SPREAD_TILE];
  __shared__ md_spread_box boxes[MD_SPREAD_MOST];
  __shared__ float theta[MD_SPREAD_MOST][2 * MD_PME_ORDER + MD_PME_ORDER][64];  // q tx, ty, tz
  __shared__ int bases[MD_SPREAD_MOST][3][64];                                  // base[0] INT_MIN: no charge
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int n[3] = {P.nx, P.ny, P.nz};
  const int S0 = blk * per, count = min(per, E.nslots / 64 - S0);
  if (wave < count) {
    const int i = E.slot_atom[(S0 + wave) * 64 + lane];
    const float q = i >= 0 ? E.param[i].w : 0.0f;
    const bool live = q != 0.0f;
    int base[3] = {0, 0, 0};
    float w[3] = {0.0f, 0.0f, 0.0f};
    if (live) md_mesh_coord(E.pos, E.np, i, P.inv, P.nx, P.ny, P.nz, base, w);
    // the stencil box: offsets of each base from the first live slot's, taken to
    // the nearest periodic representative (any representative lands on the same
    // grid points; the nearest keeps the box small)
    const uint64_t m = __ballot(live);
    const int first = m ? __ffsll((unsigned long long)m) - 1 : 0;
    for (int d = 0; d < 3; ++d) {
      const int ref = __shfl(base[d], first, 64);
      const int off = live ? md_wrap_near(base[d] - ref, n[d]) : 0;
      int lo = live ? off : INT_MAX, hi = live ? off : INT_MIN;
      for (int k = 32; k > 0; k >>= 1) {
        lo = min(lo, __shfl_xor(lo, k, 64));
        hi = max(hi, __shfl_xor(hi, k, 64));
      }
      if (lane == 0) {
        boxes[wave].ref[d] = ref;
        boxes[wave].lo[d] = lo;
        boxes[wave].hi[d] = hi;
      }
      bases[wave][d][lane] = base[d];
    }
    if (!live) bases[wave][0][lane] = INT_MIN;
    float tx[5], ty[5], tz[5];
    md_bspline5(w[0], tx, nullptr);
    md_bspline5(w[1], ty, nullptr);
    md_bspline5(w[2], tz, nullptr);
    for (int c = 0; c < 5; ++c) {
      theta[wave][c][lane] = q * tx[c];
      theta[wave][5 + c][lane] = ty[c];
      theta[wave][10 + c][lane] = tz[c];
    }
  }
  __syncthreads();
  // one pass over all of them if their joint box fits the tile
  md_spread_box box = boxes[0];
  int passes = 1, from = 0;  // a single pass starts with super-cluster `from`, the box's if it is only one's
  int shift[3] = {0, 0, 0};  // the second one's reference base from the box's
  if (count == 2) {
    const md_spread_box other = boxes[1];
    if (other.lo[0] <= other.hi[0]) {
      if (box.lo[0] > box.hi[0]) {
        box = other;
        from = 1;
      } else {
        int joint = 1;
        md_spread_box both = box;
        for (int d = 0; d < 3; ++d) {
          shift[d] = md_wrap_near(other.ref[d] - box.ref[d], n[d]);
          both.lo[d] = min(box.lo[d], other.lo[d] + shift[d]);
          both.hi[d] = max(box.hi[d], other.hi[d] + shift[d]);
          joint *= min(both.hi[d] - both.lo[d] + MD_PME_ORDER, MD_SPREAD_TILE);
          joint = min(joint, MD_SPREAD_TILE + 1);
        }
        if (joint <= MD_SPREAD_TILE) {
          box = both;
        } else {
          passes = 2;
          shift[0] = shift[1] = shift[2] = 0;
        }
      }
    }
  }
  for (int pass = 0; pass < passes; ++pass) {
    if (pass) box = boxes[pass];
    if (box.lo[0] > box.hi[0]) continue;  // no charged atom (uniform)
    int ext[3];
    for (int d = 0; d < 3; ++d) ext[d] = box.hi[d] - box.lo[d] + MD_PME_ORDER;
    const int volume = ext[0] * ext[1] * ext[2], first = passes == 2 ? pass : from, last = passes == 2 ? pass + 1 : count;
    // one super-cluster alone: with two in the pass the box fits, or the other has no charge
    if (volume > MD_SPREAD_TILE) {
      const int base[3] = {bases[first][0][lane], bases[first][1][lane], bases[first][2][lane]};
      if (base[0] == INT_MIN) continue;
      const int gx = md_wrap(base[0] + wave, P.nx);
      const float wx = theta[first][wave][lane];
      for (int b = 0; b < 5; ++b) {
        const int gy = md_wrap(base[1] + b, P.ny);
        const float wxy = wx * theta[first][5 + b][lane];
        int64_t *row = grid + ((size_t)gx * P.ny + gy) * P.nz;
        for (int c = 0; c < 5; ++c)
          md_atomic_add_i64(&row[md_wrap(base[2] + c, P.nz)], md_to_fixed(wxy * theta[first][10 + c][lane]));
      }
      continue;
    }
    for (int k = t; k < volume; k += MD_SPREAD_THREADS) tile[k] = 0;
    __syncthreads();
    for (int g = first; g < last; ++g) {
      if (bases[g][0][lane] == INT_MIN) continue;
      // the offset from its own super-cluster's reference, as its box was found
      int off[3];
      for (int d = 0; d < 3; ++d)
        off[d] = md_wrap_near(bases[g][d][lane] - boxes[g].ref[d], n[d]) + (g ? shift[d] : 0) - box.lo[d];
      const float wx = theta[g][wave][lane];
      float tz[5];
      for (int c = 0; c < 5; ++c) tz[c] = theta[g][10 + c][lane];
      unsigned long long *at = tile + ((off[0] + wave) * ext[1] + off[1]) * ext[2] + off[2];
      for (int b = 0; b < 5; ++b, at += ext[2]) {
        const float wxy = wx * theta[g][5 + b][lane];
        if (E.small_charges) {
          for (int c = 0; c < 5; ++c) atomicAdd(&at[c], (unsigned long long)md_small_to_fixed(wxy * tz[c]));
        } else {
          for (int c = 0; c < 5; ++c) atomicAdd(&at[c], (unsigned long long)md_to_fixed(wxy * tz[c]));
        }
      }
    }
    __syncthreads();
    const int x0 = md_wrap(box.ref[0] + box.lo[0], P.nx), y0 = md_wrap(box.ref[1] + box.lo[1], P.ny),
              z0 = md_wrap(box.ref[2] + box.lo[2], P.nz);
    const float inv_z = md_inverse(ext[2]), inv_y = md_inverse(ext[1]);
    // a box wider than the mesh (a stencil box of a tiny mesh) wraps more than once
    const bool once = ext[0] <= P.nx && ext[1] <= P.ny && ext[2] <= P.nz;
    for (int k = t; k < volume; k += MD_SPREAD_THREADS) {
      const long long v = (long long)tile[k];
      if (v == 0) continue;
      const int row = md_div(k, inv_z), lx = md_div(row, inv_y);
      int gx = x0 + lx, gy = y0 + row - lx * ext[1], gz = z0 + k - row * ext[2];
      if (once) {
        gx = gx >= P.nx ? gx - P.nx : gx;
        gy = gy >= P.ny ? gy - P.ny : gy;
        gz = gz >= P.nz ? gz - P.nz : gz;
      } else {
        gx %= P.nx;
        gy %= P.ny;
        gz %= P.nz;
      }
      md_atomic_add_i64(grid + ((size_t)gx * P.ny + gy) * P.nz + gz, v);
    }
    if (pass + 1 < passes) __syncthreads();  // the next pass clears the tile
  }
}

// ---- in-LDS mixed-radix Stockham transform ---------------------------------

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Where a stage finds its input and puts its output: lines of LDS (element e
// of line l at l * line + e * elem; a transposed read swaps the strides), or
// the kernel's own memory through its Ext.
struct md_fft_io {
  const float2 *in;
  int in_line, in_elem;
  float2 *out;
  int out_line;
  bool ext_in, ext_out;
};

// One Stockham stage of radix R (a compile-time constant, so a butterfly's R
// values stay in registers): output j of sub-transform k gathers the R
// inputs j + q m, multiplies input q by the twiddle w^(k q n / (ns R)) (an
// index below n, as k < ns and q < R), and takes their length-R DFT.  A stage
// that touches the kernel's memory walks it in the order of its addresses
// (Ext::line_fast: consecutive threads on consecutive lines).
template <int R, class Ext>
__device__ __forceinline__ void md_fft_stage(const md_fft_io &io, Ext &ext, int nlines, int n, int ns,
                                             const float2 *tw, float sign) {
  const int m = n / R;
  const int twstride = m / ns;
  const int dftstride = m;
  const bool lines_first = (io.ext_in || io.ext_out) && Ext::line_fast;
  const float inv = md_inverse(lines_first ? nlines : m), inv_ns = md_inverse(ns);
  for (int idx = threadIdx.x; idx < nlines * m; idx += blockDim.x) {
    const int hi = md_div(idx, inv);
    const int line = lines_first ? idx - hi * nlines : hi, j = lines_first ? hi : idx - hi * m;
    const int k = j - md_div(j, inv_ns) * ns;
    float2 v[R], o[R];
    if (io.ext_in) {
#pragma unroll
      for (int q = 0; q < R; ++q) v[q] = ext.load(line, j + q * m);
    } else {
      const float2 *src = io.in + line * io.in_line + j * io.in_elem;
#pragma unroll
      for (int q = 0; q < R; ++q) v[q] = src[q * m * io.in_elem];
    }
    if (k > 0) {
#pragma unroll
      for (int q = 1; q < R; ++q) {
        float2 w = tw[k * q * twstride];
        w.y *= -sign;  // table holds exp(-2 pi i t/n); inverse conjugates
        v[q] = cmul(v[q], w);
      }
    }
    if constexpr (R == 2) {
      o[0] = make_float2(v[0].x + v[1].x, v[0].y + v[1].y);
      o[1] = make_float2(v[0].x - v[1].x, v[0].y - v[1].y);
    } else if constexpr (R == 4) {
      float2 s0 = make_float2(v[0].x + v[2].x, v[0].y + v[2].y);
      float2 s1 = make_float2(v[0].x - v[2].x, v[0].y - v[2].y);
      float2 s2 = make_float2(v[1].x + v[3].x, v[1].y + v[3].y);
      float2 s3 = make_float2(v[1].x - v[3].x, v[1].y - v[3].y);
      // multiply s3 by sign*i: forward (-i), inverse (+i)
      float2 t3 = make_float2(-sign * s3.y, sign * s3.x);
      o[0] = make_float2(s0.x + s2.x, s0.y + s2.y);
      o[1] = make_float2(s1.x + t3.x, s1.y + t3.y);
      o[2] = make_float2(s0.x - s2.x, s0.y - s2.y);
      o[3] = make_float2(s1.x - t3.x, s1.y - t3.y);
    } else {
#pragma unroll
      for (int qo = 0; qo < R; ++qo) {
        float2 acc = v[0];
#pragma unroll
        for (int q = 1; q < R; ++q) {
          float2 w = tw[((qo * q) % R) * dftstride];
          w.y *= -sign;
          float2 p = cmul(v[q], w);
          acc.x += p.x;
          acc.y += p.y;
        }
        o[qo] = acc;
      }
    }
    const int to = (j - k) * R + k;
    if (io.ext_out) {
#pragma unroll
      for (int q = 0; q < R; ++q) ext.store(line, to + q * ns, o[q]);
    } else {
      float2 *dst = io.out + line * io.out_line + to;
#pragma unroll
      for (int q = 0; q < R; ++q) dst[q * ns] = o[q];
    }
  }
}

// pitch of a line of n values in LDS: odd, so that a transposed read of
// consecutive lines meets each bank once
__host__ __device__ inline int md_pitch(int n) { return n | 1; }

// A line pass's LDS: two buffers of `lines` lines and the twiddles.  PME_BATCH
// lines of up to 616 points fit; of more points as many as fit (15 of 640).
static size_t md_lines_lds(int n, int lines) { return sizeof(float2) * (2 * (size_t)lines * md_pitch(n) + n); }
static int md_lines(int n) {
  int lines = PME_BATCH;
  while (lines > 1 && md_lines_lds(n, lines) > PME_LDS) --lines;
  return lines;
}

// `nlines` lines of length P.n, transformed with sign -1 (forward) or +1
// (inverse) through the LDS buffers a and b.  The input is `src` (one of the
// two, with its line and element strides) or, with a null src, the kernel's
// memory through ext.load; the output is a buffer (returned, lines md_pitch
// apart) or, with `out`, the kernel's memory through ext.store.  Twiddles come
// from LDS.  Ends with a barrier unless it ends in ext.store.
template <class Ext>
__device__ __forceinline__ float2 *md_fft(float2 *a, float2 *b, const float2 *src, int line, int elem, bool out,
                                          Ext &ext, int nlines, const md_fft_plan &P, const float2 *tw, float sign) {
  const int n = P.n, pitch = md_pitch(n);
  int ns = 1;
  md_fft_io io{src, line, elem, src == a ? b : a, pitch, src == nullptr, false};
  for (int s = 0; s < P.nstages; ++s) {
    const int r = P.radix[s];
    io.ext_out = out && s + 1 == P.nstages;
    switch (r) {
      case 2: md_fft_stage<2>(io, ext, nlines, n, ns, tw, sign); break;
      case 3: md_fft_stage<3>(io, ext, nlines, n, ns, tw, sign); break;
      case 4: md_fft_stage<4>(io, ext, nlines, n, ns, tw, sign); break;
      case 5: md_fft_stage<5>(io, ext, nlines, n, ns, tw, sign); break;
      case 7: md_fft_stage<7>(io, ext, nlines, n, ns, tw, sign); break;
      case 11: md_fft_stage<11>(io, ext, nlines, n, ns, tw, sign); break;
      default: md_fft_stage<13>(io, ext, nlines, n, ns, tw, sign); break;
    }
    if (!io.ext_out) __syncthreads();
    float2 *done = io.out;
    io = md_fft_io{done, pitch, 1, done == a ? b : a, pitch, false, false};
    ns *= r;
  }
  return const_cast<float2 *>(io.in);
}

// this length's twiddles into LDS (visible after the next barrier)
__device__ __forceinline__ void md_load_twiddles(float2 *to, const md_fft_plan &P, const float2 *tw_all) {
  for (int k = threadIdx.x; k < P.n; k += blockDim.x) to[k] = tw_all[P.tw + k];
}

// The potential's rows are MD_PHI_PAD values longer than the mesh, the row's
// first values again, so an atom's five values of a row are consecutive
// wherever they start: one 16-byte and one 4-byte load, no wrapping.
typedef float md_row4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void md_row5(const float *row, float *p) {
  const md_row4 v = *reinterpret_cast<const md_row4 *>(row);
  p[0] = v.x;
  p[1] = v.y;
  p[2] = v.z;
  p[3] = v.w;
  p[4] = row[4];
}
// a value of a row, and of its continuation
__device__ __forceinline__ void md_put_phi(float *row, int z, int nz, float v) {
  row[z] = v;
  if (z < MD_PHI_PAD) row[nz + z] = v;
}

// The kernels' memory as their transforms' first and last stages see it.
//
// The charge grid's rows as lines (row r0 + line), read as f32 and cleared.
struct md_ext_charge {
  static constexpr bool line_fast = false;
  int64_t *grid;
  float2 *out;  // k_pme_z_forward's half rows
  int nz, nzc;
  __device__ float2 load(int line, int z) const {
    int64_t *p = grid + (size_t)line * nz + z;
    const int64_t v = *p;
    *p = 0;
    return make_float2((float)((double)v * 2.3283064365386963e-10), 0.0f);
  }
  __device__ void store(int line, int z, float2 v) const {
    if (z < nzc) out[(size_t)line * nzc + z] = v;
  }
};
// lines along a strided axis, `line` the consecutive index
struct md_ext_lines {
  static constexpr bool line_fast = true;
  const float2 *in;
  float2 *out;
  size_t stride;
  __device__ float2 load(int line, int e) const { return in[e * stride + line]; }
  __device__ void store(int line, int e, float2 v) const { out[e * stride + line] = v; }
};
// the Hermitian half rows of a real line (x and y are back in real space, so
// g(x, y, -kz) = conj(g(x, y, kz)) in the same row), and its real values
struct md_ext_potential {
  static constexpr bool line_fast = false;
  const float2 *in;  // the half rows: element kz of line l at l * line + kz * elem
  int line, elem;
  float *phi;
  int nz, nzc;
  __device__ float2 load(int l, int z) const {
    if (z < nzc) return in[l * line + z * elem];
    const float2 w = in[l * line + (nz - z) * elem];
    return make_float2(w.x, -w.y);
  }
  __device__ void store(int l, int z, float2 v) const { md_put_phi(phi + (size_t)l * (nz + MD_PHI_PAD), z, nz, v.x); }
};

// z pass, forward: int64 rows -> f32 -> complex FFT -> first nz/2+1 values.
// Clears the integer grid behind it.  Block = P.pz.lines rows.
__global__ void __launch_bounds__(256) k_pme_z_forward(const md_pme_table *__restrict__ T, md_bmap map) {
  extern __shared__ float2 lds[];
  int blk;
  const md_pme_table &E = md_pme_entry(T, map, blk);
  const md_pme_args &P = E.P;
  const int rows = P.nx * P.ny, lines = P.pz.lines, r0 = blk * lines, nl = min(lines, rows - r0);
  float2 *a = lds, *b = a + lines * md_pitch(P.nz), *tw = b + lines * md_pitch(P.nz);
  md_load_twiddles(tw, P.pz, P.tw);
  __syncthreads();
  md_ext_charge ext{E.grid + (size_t)r0 * P.nz, E.cgrid + (size_t)r0 * P.nzc, P.nz, P.nzc};
  md_fft(a, b, nullptr, 0, 0, true, ext, nl, P.pz, tw, -1.0f);
}

// Lines along y or x are taken a run of consecutive kz at a time, at most as
// many as a workgroup holds, the runs of one row of equal length (33 values as
// three runs of 11, not 16, 16 and 1).
static void md_set_runs(md_fft_plan &p, int nzc) {
  p.runs = (nzc + p.lines - 1) / p.lines;
  p.per = (nzc + p.runs - 1) / p.runs;
}
__device__ __forceinline__ void md_kz_run(const md_fft_plan &p, int nzc, int run, int &z0, int &nl) {
  z0 = run * p.per;
  nl = max(0, min(p.per, nzc - z0));
}

// y pass: lines along y at fixed (x, kz)
__global__ void __launch_bounds__(256) k_pme_y(const md_pme_table *__restrict__ T, md_bmap map, float sign) {
  extern __shared__ float2 lds[];
  int blk;
  const md_pme_table &E = md_pme_entry(T, map, blk);
  const md_pme_args &P = E.P;
  const int runs = P.py.runs, x = blk / runs;
  int z0, nl;
  md_kz_run(P.py, P.nzc, blk - x * runs, z0, nl);
  float2 *a = lds, *b = a + P.py.lines * md_pitch(P.ny), *tw = b + P.py.lines * md_pitch(P.ny);
  md_load_twiddles(tw, P.py, P.tw);
  __syncthreads();
  float2 *plane = E.cgrid + (size_t)x * P.ny * P.nzc + z0;
  md_ext_lines ext{plane, plane, (size_t)P.nzc};
  // (one butterfly of a single-stage plan owns its whole line, so a line is
  // read before it is written either way)
  md_fft(a, b, nullptr, 0, 0, true, ext, nl, P.py, tw, sign);
}

// x pass with the convolution: forward transform along x, multiply by the
// Ewald influence function (accumulating the energy), inverse transform.
template <bool ENERGY>
__global__ void __launch_bounds__(256) k_pme_x_convolve(const md_pme_table *__restrict__ T, md_bmap map) {
  extern __shared__ float2 lds[];
  int blk;
  const md_pme_table &E = md_pme_entry(T, map, blk);
  const md_pme_args &P = E.P;
  int64_t *energy = E.energy;
  const int runs = P.px.runs, y = blk / runs;
  int z0, nl;
  md_kz_run(P.px, P.nzc, blk - y * runs, z0, nl);
  const int pitch = md_pitch(P.nx);
  float2 *a = lds, *b = a + P.px.lines * pitch, *tw = b + P.px.lines * pitch;
  md_load_twiddles(tw, P.px, P.tw);
  __syncthreads();
  float2 *const at = E.cgrid + (size_t)y * P.nzc + z0;
  md_ext_lines ext{at, at, (size_t)P.ny * P.nzc};
  float2 *res = md_fft(a, b, nullptr, 0, 0, false, ext, nl, P.px, tw, -1.0f);
  double e = 0.0;
  int mb = y <= P.ny / 2 ? y : y - P.ny;
  const float two_pi = 6.283185307179586f;
  const float inv_nx = md_inverse(P.nx);
  for (int idx = threadIdx.x; idx < nl * P.nx; idx += blockDim.x) {
    const int l = md_div(idx, inv_nx), x = idx - l * P.nx;
    int kz = z0 + l;
    int ma = x <= P.nx / 2 ? x : x - P.nx;
    int mc = kz;
    float2 v = res[l * pitch + x];
    float2 outv = make_float2(0.0f, 0.0f);
    if (!(x == 0 && y == 0 && kz == 0)) {
      float kx = two_pi * (ma * P.invf[0]);
      float ky = two_pi * (ma * P.invf[3] + mb * P.invf[4]);
      float kzv = two_pi * (ma * P.invf[6] + mb * P.invf[7] + mc * P.invf[8]);
      float k2 = kx * kx + ky * ky + kzv * kzv;
      float mod = P.mod_x[x] * P.mod_y[y] * P.mod_z[kz];
      float factor = P.prefactor * __expf(k2 * P.exp_scale) / (k2 * mod);
      if (ENERGY) {
        // the half grid stands for both k and -k except on the kz = 0 and
        // kz = nz/2 planes, which are their own partners
        float weight = (kz == 0 || (2 * kz == P.nz)) ? 1.0f : 2.0f;
        e += (double)(weight * factor * (v.x * v.x + v.y * v.y));
      }
      outv = make_float2(2.0f * factor * v.x, 2.0f * factor * v.y);
    }
    res[l * pitch + x] = outv;
  }
  __syncthreads();
  md_fft(a, b, res, pitch, 1, true, ext, nl, P.px, tw, 1.0f);
  if (ENERGY) {
    int64_t f = md_wave_sum_i64((int64_t)rint(e * 4294967296.0));
    if ((threadIdx.x & 63) == 0) md_atomic_add_i64(energy + MD_E_RECIPROCAL, f);
  }
}

// z pass, inverse: Hermitian half line -> full line -> inverse FFT -> real.
__global__ void __launch_bounds__(256) k_pme_z_inverse(const md_pme_table *__restrict__ T, md_bmap map) {
  extern __shared__ float2 lds[];
  int blk;
  const md_pme_table &E = md_pme_entry(T, map, blk);
  const md_pme_args &P = E.P;
  const int rows = P.nx * P.ny, lines = P.pz.lines, r0 = blk * lines, nl = min(lines, rows - r0);
  float2 *a = lds, *b = a + lines * md_pitch(P.nz), *tw = b + lines * md_pitch(P.nz);
  md_load_twiddles(tw, P.pz, P.tw);
  __syncthreads();
  md_ext_potential ext{E.cgrid + (size_t)r0 * P.nzc, P.nzc, 1, E.phi + (size_t)r0 * (P.nz + MD_PHI_PAD), P.nz, P.nzc};
  md_fft(a, b, nullptr, 0, 0, true, ext, nl, P.pz, tw, 1.0f);
}

// values of one LDS buffer for a whole x-plane: ny lines along z, then nz/2+1
// along y
__host__ __device__ inline int md_plane_buffer(int ny, int nz) {
  const int rows = ny * md_pitch(nz), columns = (nz / 2 + 1) * md_pitch(ny);
  return rows > columns ? rows : columns;
}

// The z and y passes of one x-plane in one workgroup, the plane kept in LDS
// between them (meshes whose plane fits).  The same line transforms as
// k_pme_z_forward then k_pme_y, with the same inputs, so the same bits; one
// launch and one trip through memory fewer.  The first stage reads the grid
// and the last writes the spectrum; the y lines' first stage reads the z
// lines' output transposed, so nothing is copied in between.
#define MD_PLANE_THREADS 512
__global__ void __launch_bounds__(MD_PLANE_THREADS) k_pme_yz_forward(const md_pme_table *__restrict__ T, md_bmap map) {
  extern __shared__ float2 lds[];
  int x;
  const md_pme_table &E = md_pme_entry(T, map, x);
  const md_pme_args &P = E.P;
  const int ny = P.ny, nz = P.nz, nzc = P.nzc, size = md_plane_buffer(ny, nz);
  float2 *a = lds, *b = lds + size, *twz = b + size, *twy = twz + nz;
  md_load_twiddles(twz, P.pz, P.tw);
  md_load_twiddles(twy, P.py, P.tw);
  __syncthreads();
  md_ext_charge rows{E.grid + (size_t)x * ny * nz, nullptr, nz, nzc};
  float2 *res = md_fft(a, b, nullptr, 0, 0, false, rows, ny, P.pz, twz, -1.0f);  // [y][kz]
  float2 *plane = E.cgrid + (size_t)x * ny * nzc;
  md_ext_lines columns{plane, plane, (size_t)nzc};
  md_fft(a, b, res, 1, md_pitch(nz), true, columns, nzc, P.py, twy, -1.0f);  // [ky][kz]
}

// The inverse y and z passes of one x-plane (k_pme_y with +1, then
// k_pme_z_inverse), the plane kept in LDS between them.
__global__ void __launch_bounds__(MD_PLANE_THREADS) k_pme_yz_inverse(const md_pme_table *__restrict__ T, md_bmap map) {
  extern __shared__ float2 lds[];
  int x;
  const md_pme_table &E = md_pme_entry(T, map, x);
  const md_pme_args &P = E.P;
  const int ny = P.ny, nz = P.nz, nzc = P.nzc, size = md_plane_buffer(ny, nz);
  float2 *a = lds, *b = lds + size, *twz = b + size, *twy = twz + nz;
  md_load_twiddles(twz, P.pz, P.tw);
  md_load_twiddles(twy, P.py, P.tw);
  __syncthreads();
  float2 *plane = E.cgrid + (size_t)x * ny * nzc;
  md_ext_lines columns{plane, plane, (size_t)nzc};
  float2 *res = md_fft(a, b, nullptr, 0, 0, false, columns, nzc, P.py, twy, 1.0f);  // [kz][y]
  md_ext_potential rows{res, 1, md_pitch(ny), E.phi + (size_t)x * ny * (nz + MD_PHI_PAD), nz, nzc};
  float2 *free_buffer = res == a ? b : a;
  // the rows' first stage reads res through `rows`, so it writes the other
  md_fft(free_buffer, res, nullptr, 0, 0, true, rows, ny, P.pz, twz, 1.0f);
}

// Every atom's force, one thread per slot of the nonbonded list's spatial
// order: the pair kernel's i-force sums (cleared behind the read) and, as j
// atom, the force of every list entry naming its cluster, each rounded to
// Q32.32 on its own (the value an atomic per entry would add); the bonded
// terms' pieces; and dE/dQ interpolated from the mesh.  A slot is the only one
// holding its atom and integer sums have no order, so the force is written
// once, plainly, and nothing has to clear it.
//
// Bound by the latency of its dependent loads on small systems, by the L2 on
// large ones: blocks are laid out XCD by XCD, so that neighbouring slots read
// neighbouring list entries and mesh rows through one L2.  As three passes,
// each reading and writing the force, the same work took 37 us at 2,168 atoms
// (so: 15), 95 at 243k (47) and 226 on 64 replicas (168).
#define MD_FORCES_THREADS 64
__global__ void __launch_bounds__(MD_FORCES_THREADS) k_forces(const md_pme_table *__restrict__ T, md_bmap map, int energies) {
  int blk;
  const md_pme_table &E = T[md_locate(map, md_xcd_block(blockIdx.x, gridDim.x), blk)];
  const md_pme_args &P = E.P;
  const md_pair_forces &F = E.F;
  if (energies && blk == 0) {
    // the pair kernel's energy and counts: one wave, lane per part
    int64_t *part = F.part + threadIdx.x * MD_ENERGY_STRIDE;
    int64_t *const to[3] = {E.energy + MD_E_PAIR, F.census, F.blocks};
    for (int k = 0; k < 3; ++k) {
      const int64_t v = md_wave_sum_i64(part[k]);
      part[k] = 0;
      if (threadIdx.x == 0) *to[k] += v;
    }
  }
  const int np = E.np, nslots = E.nslots;
  const int s = blk * MD_FORCES_THREADS + threadIdx.x;
  const int i = E.slot_atom[s];
  int64_t f[3];
  for (int d = 0; d < 3; ++d) {
    f[d] = F.slot_force[d * nslots + s];
    F.slot_force[d * nslots + s] = 0;
  }
  if (i < 0) return;
  const float q = E.param[i].w;
  {
    // the entries naming the slot's cluster, four records in flight at a time
    const int J = s / MD_CLUSTER;
    const float *jf = F.j_force + (s - J * MD_CLUSTER) * 3;
    const int *je = F.j_entries;
    int k = F.j_start[J];
    const int end = F.j_start[J + 1];
    for (; k + 4 <= end; k += 4) {
      const float *r[4];
      float v[4][3];
#pragma unroll
      for (int u = 0; u < 4; ++u) r[u] = jf + (size_t)je[k + u] * 24;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int d = 0; d < 3; ++d) v[u][d] = r[u][d];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int d = 0; d < 3; ++d) f[d] += md_to_fixed(v[u][d]);
    }
    for (; k < end; ++k) {
      const float *e = jf + (size_t)je[k] * 24;
      for (int d = 0; d < 3; ++d) f[d] += md_to_fixed(e[d]);
    }
  }
  {
    int k = E.piece_start[i];
    const int end = E.piece_start[i + 1];
    for (; k + 4 <= end; k += 4) {
      const int64_t *t = E.piece + 3 * (size_t)k;
      for (int d = 0; d < 3; ++d) f[d] += t[d] + t[3 + d] + t[6 + d] + t[9 + d];
    }
    for (; k < end; ++k)
      for (int d = 0; d < 3; ++d) f[d] += E.piece[3 * (size_t)k + d];
  }
  if (q != 0.0f) {
    const float *phi = E.phi;
    int base[3];
    float w[3];
    md_mesh_coord(E.pos, np, i, P.inv, P.nx, P.ny, P.nz, base, w);
    float tx[5], ty[5], tz[5], dx[5], dy[5], dz[5];
    md_bspline5(w[0], tx, dx);
    md_bspline5(w[1], ty, dy);
    md_bspline5(w[2], tz, dz);
    const int pitch = P.nz + MD_PHI_PAD, gz = md_wrap_once(base[2], P.nz);
    float fx = 0.0f, fy = 0.0f, fz = 0.0f;
#pragma unroll
    for (int a = 0; a < 5; ++a) {
      const float *plane = phi + (size_t)md_wrap_once(base[0] + a, P.nx) * P.ny * pitch + gz;
      float p[5][5];
#pragma unroll
      for (int b = 0; b < 5; ++b) md_row5(plane + md_wrap_once(base[1] + b, P.ny) * pitch, p[b]);
#pragma unroll
      for (int b = 0; b < 5; ++b) {
        float sx = 0.0f, sz = 0.0f;
#pragma unroll
        for (int c = 0; c < 5; ++c) {
          sz += p[b][c] * dz[c];
          sx += p[b][c] * tz[c];
        }
        fx += dx[a] * ty[b] * sx;
        fy += tx[a] * dy[b] * sx;
        fz += tx[a] * ty[b] * sz;
      }
    }
    // d/df chain rule back to Cartesian (src/reference/forces/pme.ts:246-260)
    float dfx = -q * fx * P.nx, dfy = -q * fy * P.ny, dfz = -q * fz * P.nz;
    const float *M = P.invf;
    float Fx = dfx * M[0] + dfy * M[1] + dfz * M[2];
    float Fy = dfx * M[3] + dfy * M[4] + dfz * M[5];
    float Fz = dfx * M[6] + dfy * M[7] + dfz * M[8];
    f[0] += md_to_fixed(Fx);
    f[1] += md_to_fixed(Fy);
    f[2] += md_to_fixed(Fz);
  }
  for (int d = 0; d < 3; ++d) E.force[d * np + i] = f[d];
}

// ---- host -------------------------------------------------------------------

struct md_pme_host {
  md_fft_plan px, py, pz;
  float *mod = nullptr;  // x | y | z
  float2 *tw = nullptr;
};

static md_fft_plan make_plan(int n, int tw_offset) {
  md_fft_plan p{};
  p.n = n;
  p.tw = tw_offset;
  p.lines = md_lines(n);
  int r = n;
  // radix 4 first, then 2, 3, 5, 7, then any remaining prime (direct DFT)
  while (r % 4 == 0) {
    if (p.nstages >= PME_MAX_STAGES) break;
    p.radix[p.nstages++] = 4;
    r /= 4;
  }
  for (int f : {2, 3, 5, 7, 11, 13})
    while (r % f == 0) {
      if (p.nstages >= PME_MAX_STAGES) throw md_error(MD_ERR_NOT_SMOOTH, "mesh size has too many factors");
      p.radix[p.nstages++] = f;
      r /= f;
    }
  if (r != 1)
    throw md_error(MD_ERR_NOT_SMOOTH, std::to_string(n) + " has a prime factor above 13 (" + std::to_string(r) +
                                          " is left); PME mesh sizes must be 13-smooth");
  return p;
}

// |b(m)|^2 of the order-5 spline with the 1e-7 neighbour guard
// (src/reference/forces/bspline.ts:102-132), as its reciprocal's factor
static std::vector<double> moduli(int n) {
  const double knots[5] = {1.0 / 24, 11.0 / 24, 11.0 / 24, 1.0 / 24, 0.0};
  std::vector<double> m(n);
  for (int k = 0; k < n; ++k) {
    double re = 0, im = 0;
    for (int j = 0; j < 5 && j < n; ++j) {
      double a = 2.0 * M_PI * (double)k * j / n;
      re += knots[j] * std::cos(a);
      im += knots[j] * std::sin(a);
    }
    m[k] = re * re + im * im;
  }
  for (int k = 0; k < n; ++k)
    if (m[k] < 1e-7) m[k] = 0.5 * (m[(k - 1 + n) % n] + m[(k + 1) % n]);
  return m;
}

static md_pme_host &pme_host(md_system *s) { return *reinterpret_cast<md_pme_host *>(s->pme_ext); }

void md_pme_setup(md_system *s) {
  s->pme_ext = new md_pme_host();
  auto &H = pme_host(s);
  int nx = s->grid[0], ny = s->grid[1], nz = s->grid[2];
  s->pme_nx = nx;
  s->pme_ny = ny;
  s->pme_nz = nz;
  s->pme_nzc = nz / 2 + 1;
  int lens[3] = {nx, ny, nz};
  std::vector<float2> tw;
  int off[3];
  for (int d = 0; d < 3; ++d) {
    off[d] = (int)tw.size();
    for (int t = 0; t < lens[d]; ++t) {
      double a = -2.0 * M_PI * t / lens[d];
      tw.push_back(make_float2((float)std::cos(a), (float)std::sin(a)));
    }
  }
  H.px = make_plan(nx, off[0]);
  H.py = make_plan(ny, off[1]);
  H.pz = make_plan(nz, off[2]);
  md_set_runs(H.px, s->pme_nzc);
  md_set_runs(H.py, s->pme_nzc);
  std::vector<float> mod;
  for (int d = 0; d < 3; ++d)
    for (double v : moduli(lens[d])) mod.push_back((float)v);
  H.mod = md_alloc<float>(s, mod.size());
  H.tw = md_alloc<float2>(s, tw.size());
  MD_HIP(hipMemcpyAsync(H.mod, mod.data(), sizeof(float) * mod.size(), hipMemcpyHostToDevice, s->stream));
  MD_HIP(hipMemcpyAsync(H.tw, tw.data(), sizeof(float2) * tw.size(), hipMemcpyHostToDevice, s->stream));
  size_t g = (size_t)nx * ny * nz;
  s->pme_grid = md_alloc<int64_t>(s, g);
  s->pme_cgrid = md_alloc<float2>(s, (size_t)nx * ny * s->pme_nzc);
  s->pme_phi = md_alloc<float>(s, (size_t)nx * ny * (nz + MD_PHI_PAD));
  MD_HIP(hipStreamSynchronize(s->stream));
}

void md_pme_free(md_system *s) {
  delete reinterpret_cast<md_pme_host *>(s->pme_ext);
  s->pme_ext = nullptr;
}

// The mesh's box-dependent arguments, from a reduced box b and its
// constants: the same on the host (table set-up) and on the device (a box
// changed by the Monte Carlo barostat).
__host__ __device__ inline void md_pme_box_fields(md_pme_args &P, const double *b, const md_box &d) {
#pragma clang fp contract(off)
  for (int k = 0; k < 9; ++k) {
    P.inv[k] = d.invd[k];
    P.invf[k] = d.inv[k];
  }
  P.prefactor = (float)(MD_ONE_4PI_EPS0 * 2.0 * M_PI / md_box_volume(b));
}

static md_pme_args pme_args(md_system *s) {
  auto &H = pme_host(s);
  md_pme_args P;
  P.nx = s->pme_nx;
  P.ny = s->pme_ny;
  P.nz = s->pme_nz;
  P.nzc = s->pme_nzc;
  P.px = H.px;
  P.py = H.py;
  P.pz = H.pz;
  P.tw = H.tw;
  P.mod_x = H.mod;
  P.mod_y = H.mod + P.nx;
  P.mod_z = H.mod + P.nx + P.ny;
  md_pme_box_fields(P, s->box, s->dbox);
  P.exp_scale = (float)(-1.0 / (4.0 * s->alpha * s->alpha));
  return P;
}

static md_pme_table pme_table(md_system *s) {
  md_pme_table E;
  E.P = pme_args(s);
  E.n = s->n;
  E.np = s->np;
  E.nslots = s->nb.nslots;
  E.pos = s->pos;
  E.param = s->atom_param;
  E.slot_atom = s->slot_atom;
  E.grid = s->pme_grid;
  E.cgrid = s->pme_cgrid;
  E.phi = s->pme_phi;
  E.force = s->force;
  E.energy = s->energy;
  E.small_charges = 1;
  for (double q : s->charge)
    if (!(std::fabs(q) < MD_SMALL_FIXED)) E.small_charges = 0;
  E.F = md_nb_pair_forces(s);
  E.piece = s->term_piece;
  E.piece_start = s->atom_piece_start;
  return E;
}

struct md_pme_group {
  md_pme_table *table = nullptr;
  md_launch spread, zrows, ylines, xlines, gather, planes;
  int spread_per = 1;             // super-clusters of a spreading workgroup
  size_t lz = 0, ly = 0, lx = 0;  // dynamic LDS of the three passes
  size_t lyz = 0;                 // dynamic LDS of a whole x-plane
  bool fused_yz = false;          // the y and z passes per x-plane in one launch
};

static md_pme_group &pg(md_group *g) { return *reinterpret_cast<md_pme_group *>(g->pme); }

void md_pme_group_setup(md_group *g) {
  auto *G = new md_pme_group();
  g->pme = G;
  std::vector<int> spread, zrows, ylines, xlines, gather, planes;
  int my = 0, mz = 0;
  long supers = 0;
  for (md_system *s : g->reps) supers += s->has_nonbonded ? s->nb.nslots / 64 : 0;
  G->spread_per = supers >= MD_SPREAD_PAIRED ? 2 : 1;
  for (md_system *s : g->reps) {
    bool on = s->has_nonbonded;
    int nx = s->pme_nx, ny = s->pme_ny, nz = s->pme_nz;
    spread.push_back(on ? (s->nb.nslots / 64 + G->spread_per - 1) / G->spread_per : 0);
    zrows.push_back(on ? (nx * ny + pme_host(s).pz.lines - 1) / pme_host(s).pz.lines : 0);
    ylines.push_back(on ? nx * pme_host(s).py.runs : 0);
    xlines.push_back(on ? ny * pme_host(s).px.runs : 0);
    gather.push_back(on ? s->nb.nslots / MD_FORCES_THREADS : 0);
    planes.push_back(on ? nx : 0);
    if (on) {
      my = std::max(my, ny);
      mz = std::max(mz, nz);
      G->lx = std::max(G->lx, md_lines_lds(nx, md_lines(nx)));
      G->ly = std::max(G->ly, md_lines_lds(ny, md_lines(ny)));
      G->lz = std::max(G->lz, md_lines_lds(nz, md_lines(nz)));
    }
  }
  G->spread = md_make_launch(g, spread);
  G->zrows = md_make_launch(g, zrows);
  G->ylines = md_make_launch(g, ylines);
  G->xlines = md_make_launch(g, xlines);
  G->gather = md_make_launch(g, gather);
  G->planes = md_make_launch(g, planes);
  // planes of up to about 64^2 in LDS, two workgroups to a CU
  G->lyz = sizeof(float2) * (2 * (size_t)md_plane_buffer(my, mz) + my + mz);
  G->fused_yz = G->lyz <= 68 * 1024;
  auto allow = [](std::initializer_list<const void *> kernels, size_t lds) {
    if (lds > 64 * 1024)
      for (auto *k : kernels) MD_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  };
  allow({(const void *)k_pme_z_forward, (const void *)k_pme_z_inverse}, G->lz);
  allow({(const void *)k_pme_y}, G->ly);
  allow({(const void *)k_pme_x_convolve<true>, (const void *)k_pme_x_convolve<false>}, G->lx);
  if (G->fused_yz) allow({(const void *)k_pme_yz_forward, (const void *)k_pme_yz_inverse}, G->lyz);
  G->table = md_group_alloc<md_pme_table>(g, g->reps.size());
  md_pme_group_refresh(g);
}

void md_pme_group_refresh(md_group *g) {
  std::vector<md_pme_table> host;
  for (md_system *s : g->reps) host.push_back(s->has_nonbonded ? pme_table(s) : md_pme_table{});
  MD_HIP(hipMemcpyAsync(pg(g).table, host.data(), sizeof(md_pme_table) * host.size(), hipMemcpyHostToDevice,
                        g->stream));
  MD_HIP(hipStreamSynchronize(g->stream));
}

// Replica 0's box-dependent mesh arguments from a box in device memory (a
// barostat move).
__global__ void k_pme_box(md_pme_table *T, const double *box) {
  md_box d{};
  bool bad = false;
  md_box_from_matrix(box, d, bad);
  md_pme_box_fields(T[0].P, box, d);
}

void md_pme_box_from_device(md_group *g, const double *box) {
  k_pme_box<<<1, 1, 0, g->stream>>>(pg(g).table, box);
  MD_HIP(hipGetLastError());
}

void md_pme_group_free(md_group *g) {
  delete &pg(g);
  g->pme = nullptr;
}

void md_pme(md_group *g, bool energy, hipStream_t st) {
  auto &G = pg(g);
  if (G.spread.total == 0) return;
  const md_pme_table *T = G.table;
  k_pme_spread<<<G.spread.total, MD_SPREAD_THREADS, 0, st>>>(T, G.spread.map, G.spread_per);
  md_mark(g, MD_PHASE_FFT);
  if (G.fused_yz) {
    k_pme_yz_forward<<<G.planes.total, MD_PLANE_THREADS, G.lyz, st>>>(T, G.planes.map);
  } else {
    k_pme_z_forward<<<G.zrows.total, 256, G.lz, st>>>(T, G.zrows.map);
    k_pme_y<<<G.ylines.total, 256, G.ly, st>>>(T, G.ylines.map, -1.0f);
  }
  if (energy)
    k_pme_x_convolve<true><<<G.xlines.total, 256, G.lx, st>>>(T, G.xlines.map);
  else
    k_pme_x_convolve<false><<<G.xlines.total, 256, G.lx, st>>>(T, G.xlines.map);
  if (G.fused_yz) {
    k_pme_yz_inverse<<<G.planes.total, MD_PLANE_THREADS, G.lyz, st>>>(T, G.planes.map);
  } else {
    k_pme_y<<<G.ylines.total, 256, G.ly, st>>>(T, G.ylines.map, 1.0f);
    k_pme_z_inverse<<<G.zrows.total, 256, G.lz, st>>>(T, G.zrows.map);
  }
  MD_HIP(hipGetLastError());
}

void md_forces(md_group *g, bool energy) {
  auto &G = pg(g);
  if (G.spread.total == 0) return;
  md_mark(g, MD_PHASE_FORCES);
  k_forces<<<G.gather.total, MD_FORCES_THREADS, 0, g->stream>>>(G.table, G.gather.map, energy ? 1 : 0);
  MD_HIP(hipGetLastError());
}
