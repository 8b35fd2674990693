// Matrix-free BiCGSTAB on grid values of the same cut-cell FV discretisation.
//
// The grid-value operator of the reference (Trainer.residual_vector with
// compute_Ax_and_b_discrete_fn, jax_dips/solvers/poisson/trainer.py:883-890,
// discretization.py:522-741) is the per-point residual of the training step with
// the network replaced by values of a grid function u, read through a ghost layer
// that extrapolates linearly beyond the box (u[-1] = 2 u[0] - u[1] per axis,
// domain/interpolate.py:762-816).  The zoom-0 records of the eval grid therefore
// define it: r(p) = c_p + sum_e w_e u(p + o_e); the phase bit of an entry is
// irrelevant here because the grid function carries one value per node.
// BiCGSTAB solves A u = -c with float32 operator applications and float64
// inner products and norms, reduced deterministically (fixed block order).
#include <math.h>

#include <algorithm>
#include <utility>

#include "dips_common.h"
#include "dips_hip.h"

namespace dips {

constexpr int kJudgeThreads = 256;

// grid value with the linear ghost layer: indices -1 and n are extrapolated
__device__ __forceinline__ float u_ghost(const float* __restrict__ u, int i, int j, int k, int nx, int ny, int nz) {
  // tensor product of 1-D rules: idx in [0,n) -> itself; -1 -> 2*[0] - [1]; n -> 2*[n-1] - [n-2]
  int ia[2], ja[2], ka[2];
  float wi[2], wj[2], wk[2];
  int ni = 1, nj = 1, nk = 1;
  auto rule = [](int idx, int n, int* a, float* w, int& cnt) {
    if (idx < 0) {
      a[0] = 0, a[1] = 1, w[0] = 2.0f, w[1] = -1.0f, cnt = 2;
    } else if (idx >= n) {
      a[0] = n - 1, a[1] = n - 2, w[0] = 2.0f, w[1] = -1.0f, cnt = 2;
    } else {
      a[0] = idx, w[0] = 1.0f, cnt = 1;
    }
  };
  rule(i, nx, ia, wi, ni);
  rule(j, ny, ja, wj, nj);
  rule(k, nz, ka, wk, nk);
  float s = 0.0f;
  for (int a = 0; a < ni; ++a)
    for (int b = 0; b < nj; ++b)
      for (int c = 0; c < nk; ++c)
        s = fmaf(wi[a] * wj[b] * wk[c], u[((int64_t)ia[a] * ny + ja[b]) * nz + ka[c]], s);
  return s;
}

// Entry (w, offset) of a row at node (i, j, k): the grid value it reads, with the ghost layer.
__device__ __forceinline__ float u_entry(const float* __restrict__ u, uint32_t code, int i, int j, int k, int nx, int ny,
                                         int nz) {
  int ox, oy, oz;
  dips_decode_offset(code, ox, oy, oz);
  const int ii = i + ox, jj = j + oy, kk = k + oz;
  if (ii >= 0 && ii < nx && jj >= 0 && jj < ny && kk >= 0 && kk < nz) return u[((int64_t)ii * ny + jj) * nz + kk];
  if (ii >= -1 && ii <= nx && jj >= -1 && jj <= ny && kk >= -1 && kk <= nz) return u_ghost(u, ii, jj, kk, nx, ny, nz);
  return 0.0f;  // beyond the single ghost layer: cannot occur for stencils of radius 2 around interior points
}

// y[pt] = (with_c ? c_row : 0) + sum_e w_e u(pt + o_e) for every record row, each row's entries in order.
// Bound by the records' bytes (8 per entry: 118 MB and 25 us at 128^3).  One lane owns a row and adds its
// entries, but kApplyPer lanes fetch them: a wavefront's load instruction reads 8 rows' next 8 entries (whole
// lines) instead of one entry of each of 64 rows, all of a round's loads are issued before the first use, and
// (w, u) reach the owner through LDS.  At 128^3 (star, 15 M entries): 96 us with a lane per row reading its own
// entries one by one, 57 us with 8 of them in flight, 39 us like this.
// Workgroups take the rows from the last on, since the records end with their longest rows (33 entries on
// average next to the interface), which would else start last: 72 against 58 us.  Of each kRowGroup workgroups
// every die takes neighbours, whose rows read the same u (64 workgroups: 39 us, 128: 40, 512: 58, as one die then
// has all the long rows).
// stop (null, or a flag the solver's kernels raise): nothing is done once it is nonzero.
constexpr int kXcds = 8;
constexpr int kRowGroup = 64;
constexpr int kApplyPer = 8;                          // entries of a row per round: a bulk row has 7
constexpr int kApplyPasses = kApplyPer;               // load instructions per round, 64 / kApplyPer rows each
constexpr int kPassRows = DIPS_WAVE / kApplyPer;
__global__ __launch_bounds__(kJudgeThreads) void grid_apply_kernel(
    int nx, int ny, int nz, const int32_t* __restrict__ row_point, const int32_t* __restrict__ row_ptr,
    const float* __restrict__ row_c, int64_t nrows, const uint32_t* __restrict__ ent_code,
    const float* __restrict__ ent_w, int64_t nnz, const float* __restrict__ u, float* __restrict__ y, int with_c,
    const double* __restrict__ stop) {
  if (stop && *stop != 0.0) return;
  __shared__ int4 rows[kJudgeThreads / DIPS_WAVE][DIPS_WAVE];  // point, first entry, entries, whether no ghost is read
  __shared__ float2 wu[kJudgeThreads / DIPS_WAVE][DIPS_WAVE * (kApplyPer + 1)];  // per row, padded by one
  const int lane = threadIdx.x & (DIPS_WAVE - 1), wave = threadIdx.x / DIPS_WAVE;
  const int64_t back = (int64_t)gridDim.x - 1 - blockIdx.x, base = back / kRowGroup * kRowGroup, in = back - base;
  const int64_t blk =
      base + kRowGroup <= (int64_t)gridDim.x ? base + (in % kXcds) * (kRowGroup / kXcds) + in / kXcds : back;
  const int64_t row = blk * kJudgeThreads + threadIdx.x;
  const int64_t npts = (int64_t)nx * ny * nz;
  int pt = -1, beg = 0;
  uint32_t len = 0;  // entries are counted from their row's first: entry indices go up to the largest int
  if (row < nrows) {
    pt = row_point[row];
    beg = max(row_ptr[row], 0);
    len = (uint32_t)max(min((int64_t)row_ptr[row + 1], nnz) - beg, (int64_t)0);
  }
  const bool on = pt >= 0 && pt < npts;
  if (!on) len = 0;
  {
    // two nodes inside the grid (three below the top of the last axis: codes 125..127, outside the 5^3 cube,
    // decode to 3 there)
    const int k = pt % nz, ij = pt / nz, j = ij % ny, i = ij / ny;
    const bool inner = on && i >= 2 && i < nx - 2 && j >= 2 && j < ny - 2 && k >= 2 && k < nz - 3;
    rows[wave][lane] = make_int4(pt, beg, (int)len, inner ? 1 : 0);
  }
  float acc = (on && with_c) ? row_c[row] : 0.0f;
  const int sub = lane % kApplyPer, slot = lane / kApplyPer;
  __builtin_amdgcn_wave_barrier();
  for (uint32_t c0 = 0; __any(c0 < len); c0 += kApplyPer) {
    int4 rw[kApplyPasses];
    uint32_t code[kApplyPasses];
    float w[kApplyPasses], v[kApplyPasses];
#pragma unroll
    for (int q = 0; q < kApplyPasses; ++q) {
      rw[q] = rows[wave][q * kPassRows + slot];
      code[q] = 0;
      w[q] = 0.0f;
      if (c0 + sub < (uint32_t)rw[q].z) {
        const uint32_t e = (uint32_t)rw[q].y + c0 + sub;
        code[q] = ent_code[e];
        w[q] = ent_w[e];
      }
    }
#pragma unroll
    for (int q = 0; q < kApplyPasses; ++q) {
      v[q] = 0.0f;
      if (c0 + sub < (uint32_t)rw[q].z) {
        if (rw[q].w) {
          int ox, oy, oz;
          dips_decode_offset(code[q], ox, oy, oz);
          v[q] = u[(int64_t)rw[q].x + ((int64_t)ox * ny + oy) * nz + oz];
        } else {
          const int p = rw[q].x, ij = p / nz;
          v[q] = u_entry(u, code[q], ij / ny, ij % ny, p % nz, nx, ny, nz);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < kApplyPasses; ++q)
      wu[wave][(q * kPassRows + slot) * (kApplyPer + 1) + sub] = make_float2(w[q], v[q]);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < kApplyPer; ++q) {
      const float2 p = wu[wave][lane * (kApplyPer + 1) + q];
      if (c0 + q < len) acc = fmaf(p.x, p.y, acc);
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (on) y[pt] = acc;
}

// dst = a*x + b*y + c*z (any pointer may alias dst; null operands count as zero)
__global__ void axpbypcz_kernel(int64_t n, float* dst, double a, const float* x, double b, const float* y,
                                double c, const float* z) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  double v = 0.0;
  if (x) v += a * (double)x[t];
  if (y) v += b * (double)y[t];
  if (z) v += c * (double)z[t];
  dst[t] = (float)v;
}

// Inner products: element t belongs to thread t mod (kDotBlocks kJudgeThreads), which adds its elements in
// order; a wavefront's threads are added in a fixed tree, a workgroup's wavefronts in order, and the
// workgroups' partial sums in order (ordered_sum).  Every kernel below that forms one keeps this order.
// Workgroups past the last element would add zeros and are not launched (dot_blocks).
constexpr int kDotBlocks = 512;
constexpr int64_t kDotStride = (int64_t)kDotBlocks * kJudgeThreads;
static int dot_blocks(int64_t n) { return (int)std::min<int64_t>(kDotBlocks, (n + kJudgeThreads - 1) / kJudgeThreads); }

// the workgroup's partial sum of s (one value per thread) to *out
__device__ __forceinline__ void block_sum(double s, double* __restrict__ out) {
  s = dips_wave_sum_d(s);
  __shared__ double red[kJudgeThreads / DIPS_WAVE];
  __syncthreads();  // the previous sum's values have been read
  if ((threadIdx.x & (DIPS_WAVE - 1)) == 0) red[threadIdx.x / DIPS_WAVE] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kJudgeThreads / DIPS_WAVE; ++w) t += red[w];
    *out = t;
  }
}

// a = sum of pa[0, nb), b = sum of pb[0, nb) in order (pb may be null), in every thread.  The additions are a
// serial chain by definition; the values come through LDS, so that the chain waits for no memory
// (one thread that read them from memory itself took 34 us for 512 values).
__device__ __forceinline__ void ordered_sum(const double* __restrict__ pa, const double* __restrict__ pb, int nb,
                                            double& a, double& b) {
  __shared__ double vals[2][kDotBlocks];
  __shared__ double tot[2];
  for (int i = threadIdx.x; i < nb; i += kJudgeThreads) {
    vals[0][i] = pa[i];
    if (pb) vals[1][i] = pb[i];
  }
  __syncthreads();
  const int w = threadIdx.x / DIPS_WAVE;
  if ((threadIdx.x & (DIPS_WAVE - 1)) == 0 && (w == 0 || (w == 1 && pb))) {
    double t = 0.0;
#pragma unroll 16
    for (int i = 0; i < nb; ++i) t += vals[w][i];
    tot[w] = t;
  }
  __syncthreads();
  a = tot[0];
  b = pb ? tot[1] : 0.0;
}

// partial[blk] = the workgroup's part of x . y and, with z, partial2[blk] that of x . z
__global__ __launch_bounds__(kJudgeThreads) void dot_partial_kernel(int64_t n, const float* __restrict__ x,
                                                                    const float* __restrict__ y,
                                                                    double* __restrict__ partial,
                                                                    const float* __restrict__ z,
                                                                    double* __restrict__ partial2,
                                                                    const double* __restrict__ stop) {
  if (stop && *stop != 0.0) return;
  double s = 0.0, s2 = 0.0;
#pragma unroll 4
  for (int64_t t = (int64_t)blockIdx.x * kJudgeThreads + threadIdx.x; t < n; t += kDotStride) {
    s = fma((double)x[t], (double)y[t], s);
    if (z) s2 = fma((double)x[t], (double)z[t], s2);
  }
  block_sum(s, partial + blockIdx.x);
  if (z) block_sum(s2, partial2 + blockIdx.x);
}

// out[slot] = sum of partial[0..nblk) in block order
__global__ __launch_bounds__(kJudgeThreads) void dot_final_kernel(const double* __restrict__ partial, int nblk,
                                                                  double* __restrict__ out, int slot) {
  double a, b;
  ordered_sum(partial, nullptr, nblk, a, b);
  if (threadIdx.x == 0) out[slot] = a;
}

// ---- one BiCGSTAB iteration on the device ------------------------------------------
// The iteration's scalars stay in device memory (the eight doubles behind the partial sums), so that the
// host waits once per kChunk iterations instead of four times in each, and every vector update also forms the
// inner products of what it has just computed: 7 launches an iteration, against 20 launches and 4 host waits
// (at 128^3: 0.50 -> 0.16 ms an iteration, of which the two operator applications take 78 us).
// A kernel sums the previous kernel's partial sums itself, in every workgroup.  Once an iteration may not
// begin (converged, or a breakdown) S[kDone] is raised and the kernels that are still queued do nothing.
// Slots are written by workgroup 0 only, and never one that another workgroup of the same kernel
// reads, except kDone, whose value decides nothing there that the partial sums do not.
enum { kRho0 = 0, kRho1 = 1, kAlpha = 2, kOmega = 3, kDone = 4, kIters = 5, kSlots = 8 };
constexpr int kChunk = 8;  // iterations between two looks at S[kDone]

struct IterArgs {
  int64_t n;
  int nb;       // workgroups, and partial sums of an inner product
  double* S;    // slots
  double* pa;   // partial sums: rh . v, then t . s
  double* ptt;  // t . t
  double* prr;  // r . r
  double* prho; // rh . r
};

// S[kDone] as one value for the whole workgroup, in the kernels whose workgroup 0 may raise it while others read it
__device__ __forceinline__ bool stopped(const double* __restrict__ S) {
  __shared__ double d;
  if (threadIdx.x == 0) d = S[kDone];
  __syncthreads();
  return d != 0.0;
}

// rh = r, p = v = 0, scalars 1; partial sums of rh . r
__global__ __launch_bounds__(kJudgeThreads) void bicg_start_kernel(IterArgs A, const float* __restrict__ r,
                                                                   float* __restrict__ rh, float* __restrict__ p,
                                                                   float* __restrict__ v) {
  double s = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * kJudgeThreads + threadIdx.x; t < A.n; t += kDotStride) {
    const float x = (float)fma(1.0, (double)r[t], 0.0);
    rh[t] = x;
    p[t] = 0.0f;
    v[t] = 0.0f;
    s = fma((double)x, (double)r[t], s);
  }
  block_sum(s, A.prho + blockIdx.x);
  if (blockIdx.x == 0 && threadIdx.x < kSlots)
    A.S[threadIdx.x] = (threadIdx.x <= kOmega) ? 1.0 : 0.0;
}

// whether the iteration begins (first: the host has tested), then p = r + beta (p - omega v)
__global__ __launch_bounds__(kJudgeThreads) void bicg_p_kernel(IterArgs A, int parity, int first, double bnorm,
                                                               double rtol, const float* __restrict__ r,
                                                               float* __restrict__ p, const float* __restrict__ v) {
  if (stopped(A.S)) return;
  const double rho = A.S[parity], alpha = A.S[kAlpha], omega = A.S[kOmega];
  double rho_new, rr;
  ordered_sum(A.prho, first ? nullptr : A.prr, A.nb, rho_new, rr);
  const bool go = (first || sqrt(rr) / bnorm > rtol) && !(rho_new == 0.0 || omega == 0.0);
  if (!go) {
    if (blockIdx.x == 0 && threadIdx.x == 0) A.S[kDone] = 1.0;
    return;
  }
  const double beta = (rho_new / rho) * (alpha / omega);
  const double c = -beta * omega;
  if (blockIdx.x == 0 && threadIdx.x == 0) A.S[parity ^ 1] = rho_new;
#pragma unroll 4
  for (int64_t t = (int64_t)blockIdx.x * kJudgeThreads + threadIdx.x; t < A.n; t += kDotStride)
    p[t] = (float)fma(c, (double)v[t], fma(beta, (double)p[t], fma(1.0, (double)r[t], 0.0)));
}

// alpha = rho / rh . v, s = r - alpha v
__global__ __launch_bounds__(kJudgeThreads) void bicg_s_kernel(IterArgs A, int parity, const float* __restrict__ r,
                                                               const float* __restrict__ v, float* __restrict__ s) {
  if (stopped(A.S)) return;
  double rhv, unused;
  ordered_sum(A.pa, nullptr, A.nb, rhv, unused);
  if (rhv == 0.0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) A.S[kDone] = 1.0;
    return;
  }
  const double alpha = A.S[parity ^ 1] / rhv;
  if (blockIdx.x == 0 && threadIdx.x == 0) A.S[kAlpha] = alpha;
#pragma unroll 4
  for (int64_t t = (int64_t)blockIdx.x * kJudgeThreads + threadIdx.x; t < A.n; t += kDotStride)
    s[t] = (float)fma(-alpha, (double)v[t], fma(1.0, (double)r[t], 0.0));
}

// omega = t . s / t . t, x += alpha p + omega s, s <- s - omega t (the next r); partial sums of r . r and rh . r
__global__ __launch_bounds__(kJudgeThreads) void bicg_x_kernel(IterArgs A, float* __restrict__ x,
                                                               const float* __restrict__ p, float* __restrict__ s,
                                                               const float* __restrict__ t_,
                                                               const float* __restrict__ rh) {
  if (A.S[kDone] != 0.0) return;
  const double alpha = A.S[kAlpha];
  double ts, tt;
  ordered_sum(A.pa, A.ptt, A.nb, ts, tt);
  const double omega = (tt > 0.0) ? ts / tt : 0.0;
  double rr = 0.0, rho = 0.0;
#pragma unroll 2
  for (int64_t t = (int64_t)blockIdx.x * kJudgeThreads + threadIdx.x; t < A.n; t += kDotStride) {
    const double sv = (double)s[t];
    x[t] = (float)fma(omega, sv, fma(alpha, (double)p[t], fma(1.0, (double)x[t], 0.0)));
    const float r = (float)fma(-omega, (double)t_[t], fma(1.0, sv, 0.0));
    s[t] = r;
    rr = fma((double)r, (double)r, rr);
    rho = fma((double)rh[t], (double)r, rho);
  }
  block_sum(rr, A.prr + blockIdx.x);
  block_sum(rho, A.prho + blockIdx.x);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    A.S[kOmega] = omega;
    A.S[kIters] += 1.0;
  }
}

struct JudgeCtx {
  const dips_grid_t* g;
  const dips_records_t* rec;
  hipStream_t st;
  double* dpart;  // kDotBlocks
  double* dres;   // kSlots result slots
};

static int apply(const JudgeCtx& C, const float* u, float* y, int with_c, const double* stop = nullptr) {
  const int64_t nb = (C.rec->nrows + kJudgeThreads - 1) / kJudgeThreads;
  hipLaunchKernelGGL(grid_apply_kernel, dim3((unsigned)nb), dim3(kJudgeThreads), 0, C.st, C.g->nx, C.g->ny, C.g->nz,
                     C.rec->row_point, C.rec->row_ptr, C.rec->row_c, C.rec->nrows, C.rec->ent_code, C.rec->ent_w,
                     C.rec->nnz, u, y, with_c, stop);
  return hip_status(hipGetLastError(), "grid_apply_kernel launch");
}

static void lin(const JudgeCtx& C, int64_t n, float* dst, double a, const float* x, double b, const float* y, double c,
                const float* z) {
  hipLaunchKernelGGL(axpbypcz_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, C.st, n, dst, a, x, b, y, c, z);
}

static void dot(const JudgeCtx& C, int64_t n, const float* x, const float* y, int slot) {
  hipLaunchKernelGGL(dot_partial_kernel, dim3(dot_blocks(n)), dim3(kJudgeThreads), 0, C.st, n, x, y, C.dpart,
                     (const float*)nullptr, (double*)nullptr, (const double*)nullptr);
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kJudgeThreads), 0, C.st, C.dpart, dot_blocks(n), C.dres, slot);
}

static int fetch(const JudgeCtx& C, double* host, int count) {
  hipError_t e = hipMemcpyAsync(host, C.dres, sizeof(double) * count, hipMemcpyDeviceToHost, C.st);
  if (e == hipSuccess) e = hipStreamSynchronize(C.st);
  return hip_status(e, "judge scalar readback");
}

int grid_apply(const dips_grid_t* g, const dips_records_t* rec, const float* u, float* y, int with_c,
               hipStream_t st) {
  JudgeCtx C{g, rec, st, nullptr, nullptr};
  return apply(C, u, y, with_c);
}

int bicgstab(const dips_grid_t* g, const dips_records_t* rec, float* x, float* work, double* dwork, int max_iter,
             double rtol, int* iters, double* relres, hipStream_t st) {
  const int64_t n = (int64_t)g->nx * g->ny * g->nz;
  float* r = work;
  float* rh = work + n;
  float* p = work + 2 * n;
  float* v = work + 3 * n;
  float* s = work + 4 * n;
  float* t = work + 5 * n;
  JudgeCtx C{g, rec, st, dwork, dwork + kDotBlocks};
  double h[kSlots];
  int status;
  // r = b - A x = -(A x + c); b = -c
  if ((status = apply(C, x, r, 1))) return status;
  lin(C, n, r, -1.0, r, 0.0, nullptr, 0.0, nullptr);
  // ||b||
  if ((status = apply(C, x, t, 0))) return status;      // t = A x
  lin(C, n, s, -1.0, r, -1.0, t, 0.0, nullptr);          // s = -(r + A x) = c
  dot(C, n, s, s, 0);
  dot(C, n, r, r, 1);
  if ((status = fetch(C, h, 2))) return status;
  const double bnorm = sqrt(h[0]) > 0 ? sqrt(h[0]) : 1.0;
  const double res = sqrt(h[1]) / bnorm;
  int it = 0;
  if (max_iter > 0 && res > rtol) {
    const int nb = dot_blocks(n);
    const dim3 grid(nb), block(kJudgeThreads);
    double* S = C.dres;
    // Three more sets of partial sums than the float64 workspace has room for at more than 128 workgroups:
    // they go to whichever of r and s is dead.  r is, from the update that makes s out of it to the end of the
    // iteration, where the next r replaces s in place and the two change names; the sums written
    // there last are read by the next iteration's first kernel, before s is written again.
    auto sums = [&](float* dead, int k) {
      if (4 * nb <= kDotBlocks) return dwork + (k + 1) * nb;
      return reinterpret_cast<double*>((reinterpret_cast<uintptr_t>(dead) + 7) & ~(uintptr_t)7) + k * nb;
    };
    IterArgs A{n, nb, S, dwork, sums(r, 0), sums(r, 1), sums(s, 2)};
    hipLaunchKernelGGL(bicg_start_kernel, grid, block, 0, st, A, r, rh, p, v);
    int parity = 0, launched = 0;
    bool done = false;
    while (!done && launched < max_iter) {
      const int chunk = std::min(kChunk, max_iter - launched);
      for (int q = 0; q < chunk; ++q, ++launched, parity ^= 1) {
        hipLaunchKernelGGL(bicg_p_kernel, grid, block, 0, st, A, parity, launched == 0 ? 1 : 0, bnorm, rtol, r, p, v);
        if ((status = apply(C, p, v, 0, S + kDone))) return status;  // v = A p
        hipLaunchKernelGGL(dot_partial_kernel, grid, block, 0, st, n, rh, v, A.pa, (const float*)nullptr,
                           (double*)nullptr, S + kDone);
        hipLaunchKernelGGL(bicg_s_kernel, grid, block, 0, st, A, parity, r, v, s);
        if ((status = apply(C, s, t, 0, S + kDone))) return status;  // t = A s
        A.ptt = sums(r, 0), A.prr = sums(r, 1), A.prho = sums(r, 2);
        hipLaunchKernelGGL(dot_partial_kernel, grid, block, 0, st, n, t, s, A.pa, t, A.ptt, S + kDone);
        hipLaunchKernelGGL(bicg_x_kernel, grid, block, 0, st, A, x, p, s, t, rh);
        std::swap(r, s);
      }
      if ((status = hip_status(hipGetLastError(), "BiCGSTAB kernels launch"))) return status;
      if ((status = fetch(C, h, kSlots))) return status;
      done = h[kDone] != 0.0;
      it = (int)h[kIters];
    }
  }
  // true residual of the float32 iterate
  if ((status = apply(C, x, t, 1))) return status;
  dot(C, n, t, t, 0);
  if ((status = fetch(C, h, 1))) return status;
  *iters = it;
  *relres = sqrt(h[0]) / bnorm;
  return DIPS_OK;
}

}  // namespace dips
