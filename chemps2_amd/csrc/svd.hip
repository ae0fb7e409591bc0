// Singular value decompositions of Split's centre sectors, all sectors of a site at once.
//
// A (m x n, m >= n; the transposed sector matrix when that is wide) = Q R after its columns
// are sorted by falling norm (Householder QR in panels of 16 columns); then one-sided
// (Hestenes) Jacobi on X = R^T: X J = Ux Sigma, so that A P = (Q J) Sigma Ux^T. Jacobi on
// the transposed triangular factor of the sorted matrix needs 7-10 sweeps where Jacobi on
// A needs 16-27 (Drmac & Veselic, SIAM J. Matrix Anal. Appl. 29 (2008) 1322 and 1343; sweep
// counts of sector matrices of 138-440 columns whose singular values span 7-9 decades), it
// works on n x n instead of m x n, and Q J is orthonormal whatever the singular values are.
//
// What bounds it is the chain of rotation rounds: a sweep is n - 1 rounds, one after the
// other, of little work each. The columns go in blocks of 16; a launch takes one round of
// block pairs, a workgroup per pair (k_svd_round): the pair's 32 x 32 Gram matrix on the
// matrix cores, the rotations of its columns on that matrix in LDS (0.2 us a round, where
// rotating the columns themselves in LDS took 1.3 us at n = 147), and the columns of X and J
// times the accumulated rotations on the matrix cores. A Gram matrix fresh from the columns
// starts every visit, so what its updates lose in small entries the next visit corrects, and
// the test that ends the sweeps (no entry above the rounding floor) is on fresh ones.
//
// Measured on the MI355X (Split and Join of one site): 196 sectors of up to 147 columns
// (L = 32, D = 2000, D2h) 3.7 ms, where one workgroup per sector rotating columns in global
// memory took 33 ms; 69 sectors of up to 615 columns (no point group, D = 2000) 20.2 ms,
// where those above 256 went to rocSOLVER's dgesvdj (930 ms). The re-joined object is 2.8e-15
// (wide: 6.0e-15) from LAPACK's, those paths' 3.1e-14 (2.2e-13).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "chm_internal.hpp"
#include "dbuf.hpp"

namespace chm {

namespace {

static_assert(SVD_ALONE == 32, "two blocks of 16");

typedef double svd_t4 __attribute__((ext_vector_type(4)));

constexpr double SVD_EPS = 1.1102230246251565e-16;  // 2^-53
constexpr int JT = 1024, JW = JT / 64;              // threads and wavefronts of the per-sector kernels
constexpr int RT = 512, RW = RT / 64;               // of the Jacobi rounds
constexpr int QT = 512, QW = QT / 64;               // of the QR kernels
constexpr int PB = 16;                              // columns of a QR panel or a Jacobi block

// sum over the wavefront (the same order for every lane; uniform result): lanes of 16 by
// DPP, the four groups through scalar registers
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return v + __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ double lane_of(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0xB1>(v);   // lane ^ 1
  v = dpp_add<0x4E>(v);   // lane ^ 2
  v = dpp_add<0x141>(v);  // the other quad of 8 lanes
  v = dpp_add<0x140>(v);  // the other 8 of 16 lanes
  return (lane_of(v, 0) + lane_of(v, 16)) + (lane_of(v, 32) + lane_of(v, 48));
}

// Round r of a round-robin over n2 (even) slots: pair k = (p, q), p < q.
__device__ __forceinline__ void pair_of(int n2, int r, int k, int& p, int& q) {
  p = (k == 0) ? 0 : ((k - 1 + r) % (n2 - 1)) + 1;
  q = ((n2 - 2 - k + r) % (n2 - 1)) + 1;
  if (p > q) { const int t = p; p = q; q = t; }
}

// The largest element's magnitude for the whole workgroup (SVD_INF when one is not finite).
constexpr double SVD_INF = __builtin_huge_val();
__device__ double max_abs(const double* __restrict__ a, int n, int tid, double* red) {
  double mx = 0.0;
  for (int e = tid; e < n; e += JT) {
    const double v = fabs(a[e]);
    mx = v <= 1.7976931348623157e308 ? fmax(mx, v) : SVD_INF;
    if (mx == SVD_INF) break;
  }
  red[tid] = mx;
  __syncthreads();
  for (int h = JT / 2; h > 0; h >>= 1) {
    if (tid < h) red[tid] = fmax(red[tid], red[tid + h]);
    __syncthreads();
  }
  mx = red[0];
  __syncthreads();
  return mx;
}

// The power of two that brings the sector to order one, column norms of A so scaled, their order
// (perm: sorted position -> column), the floor, counters cleared. One workgroup per sector. The
// rotations multiply squared norms, which takes them out of the range of doubles for columns
// below 1e-80 or above 1e77; the scale comes from the sum of the squares, or from the largest
// element where the squares themselves leave that range. A sector with an element that is
// not finite counts as zero (scale 0).
__global__ __launch_bounds__(JT) void k_svd_sort(const DevSvd* __restrict__ jobs) {
  __shared__ double nrm[SVD_MAXM], red[JT];
  const DevSvd it = jobs[blockIdx.x];
  const int m = it.m, n = it.n, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  auto norms = [&](double scale) {  // and the sum of their squares
    for (int j = wv; j < n; j += JW) {
      double s = 0.0;
      for (int i = lane; i < m; i += 64) {
        const double v = it.A[i + (size_t)m * j] * scale;
        s = fma(v, v, s);
      }
      s = wave_sum(s);
      if (lane == 0) nrm[j] = s;
    }
    __syncthreads();
    double s = 0.0;
    for (int j = lane; j < n; j += 64) s += nrm[j];
    return wave_sum(s);
  };
  double sum = norms(1.0), scale, unit = 1.0;  // unit: the scale of nrm and sum
  if (sum > 1e-200 && sum < 1e200) {
    scale = ldexp(1.0, -ilogb(sum) / 2);
  } else {
    const double mx = max_abs(it.A, m * n, tid, red);
    if (mx > 0.0 && mx < SVD_INF) {
      scale = unit = ldexp(1.0, max(-1000, min(1000, -ilogb(mx))));
      sum = norms(unit);
    } else {
      scale = mx > 0.0 ? 0.0 : 1.0;
      sum = 0.0;
      for (int j = tid; j < n; j += JT) nrm[j] = 0.0;
      __syncthreads();
    }
  }
  for (int j = tid; j < n; j += JT) {
    int r = 0;
    for (int k = 0; k < n; k++) r += (nrm[k] > nrm[j] || (nrm[k] == nrm[j] && k < j)) ? 1 : 0;
    it.perm[r] = j;
  }
  if (tid == JT - 1) {
    const double f = unit == scale ? 1.0 : scale;
    it.floor2[0] = SVD_EPS * SVD_EPS * (sum * f * f);
    it.floor2[1] = scale;
  }
  for (int q = tid; q < SVD_SWEEPS; q += JT) it.rot[q] = 0;
  if (tid == 0) *it.info = 0;
}

// W = A in sorted order and scaled, X cleared, J the identity; SVD_CHUNKS workgroups per sector.
constexpr int SVD_CHUNKS = 16;
__global__ __launch_bounds__(QT) void k_svd_copy(const DevSvd* __restrict__ jobs) {
  const DevSvd it = jobs[blockIdx.y];
  const int m = it.m, n = it.n, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const double scale = it.floor2[1];
  for (int t = blockIdx.x * QW + wv; t < n; t += SVD_CHUNKS * QW) {
    const double* a = it.A + (size_t)m * it.perm[t];
    for (int i = lane; i < m; i += 64) it.W[i + (size_t)m * t] = scale == 0.0 ? 0.0 : a[i] * scale;
    for (int i = lane; i < n; i += 64) {
      it.X[i + (size_t)n * t] = 0.0;
      it.J[i + (size_t)n * t] = i == t ? 1.0 : 0.0;
    }
  }
}

// part[w] (16 x 16 each, [i][j]) -> out[i][j] = sum over the wavefronts, in order
__device__ __forceinline__ void sum_parts(const double (*part)[256], double* out, int tid) {
  if (tid < 256) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < QW; w++) s += part[w][tid];
    out[tid] = s;
  }
}

// Step k of the QR of W: a workgroup per column block j >= k applies the reflectors of panel
// k - 1 (I - V T^T V^T), whose rows of R then go to X = R^T; the workgroup of block k also
// factors it as the next panel: V (unit lower trapezoidal, zeros above) to A, T to T, its R
// to X. The products are 16 x 16 results on the matrix cores, rows dealt out to the
// wavefronts; the panel is in LDS, or (TALL: sectors of more than SVD_MAXM rows, the others in
// the launch without TALL) factored where it lies, in W.
template <bool TALL>
__global__ __launch_bounds__(QT) void k_qr_step(const DevSvd* __restrict__ jobs, int k) {
  extern __shared__ double panel[];
  __shared__ double part[QW][256];
  __shared__ double w1[256], w2[256];
  __shared__ double tau[PB], scl[PB], bet[PB];
  const DevSvd it = jobs[blockIdx.y];
  const int m = it.m, n = it.n, nb = (n + PB - 1) / PB, j = k + (int)blockIdx.x;
  if (j >= nb || (m > SVD_MAXM) != TALL) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, lr = lane & 15, lg = lane >> 4;
  const int c0 = PB * j, cw = min(PB, n - c0);
  double* C = it.W + (size_t)m * c0;
  if (k > 0) {
    const int r0 = PB * (k - 1);
    const double* V = it.A + (size_t)m * r0;
    const double* T = it.T + 256 * (k - 1);
    svd_t4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int base = r0 + 16 * wv; base < m; base += 16 * QW) {
      double v[4], c[4];
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int row = base + 4 * lg + s;
        v[s] = row < m ? V[row + (size_t)m * lr] : 0.0;
        c[s] = (row < m && lr < cw) ? C[row + (size_t)m * lr] : 0.0;
      }
#pragma unroll
      for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v[s], c[s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) part[wv][(4 * r + lg) * 16 + lr] = acc[r];
    __syncthreads();
    sum_parts(part, w1, tid);
    __syncthreads();
    if (tid < 256) {
      const int i = tid >> 4, q = tid & 15;
      double s = 0.0;
      for (int l = 0; l <= i; l++) s = fma(T[l + 16 * i], w1[16 * l + q], s);
      w2[tid] = s;
    }
    __syncthreads();
    for (int base = r0 + 16 * wv; base < m; base += 16 * QW) {
      const int row = base + lr;
      svd_t4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const double v = row < m ? V[row + (size_t)m * (4 * s + lg)] : 0.0;
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(w2[16 * (4 * s + lg) + lr], v, d, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int c = 4 * r + lg;
        if (row < m && c < cw) {
          const double x = C[row + (size_t)m * c] - d[r];
          C[row + (size_t)m * c] = x;
          if (base == r0) it.X[c0 + c + (size_t)n * row] = x;
        }
      }
    }
  }
  if (j != k) return;
  const int q0 = PB * k, mk = m - q0;
  double* P;         // panel: column c at P + c ps
  const int ps = TALL ? m : mk;
  __syncthreads();
  if constexpr (TALL) {
    P = C + q0;
  } else {
    P = panel;
    for (int c = wv; c < PB; c += QW)
      for (int i = lane; i < mk; i += 64) P[c * ps + i] = c < cw ? C[q0 + i + (size_t)m * c] : 0.0;
    __syncthreads();
  }
  for (int c = 0; c < cw; c++) {
    double s = 0.0;
    for (int i = c + 1 + lane; i < mk; i += 64) s = fma(P[c * ps + i], P[c * ps + i], s);
    s = wave_sum(s);
    const double a = P[c * ps + c];
    double tc = 0.0, sc = 0.0, bc = a;
    if (s > 0.0) {
      bc = a >= 0.0 ? -sqrt(fma(a, a, s)) : sqrt(fma(a, a, s));
      tc = (bc - a) / bc;
      sc = 1.0 / (a - bc);
    }
    if (tid == 0) { tau[c] = tc; scl[c] = sc; bet[c] = bc; }
    for (int q = c + 1 + wv; q < cw; q += QW) {
      double d = 0.0;
      for (int i = c + 1 + lane; i < mk; i += 64) d = fma(P[c * ps + i], P[q * ps + i], d);
      d = tc * fma(sc, wave_sum(d), P[q * ps + c]);
      const double ds = d * sc;
      for (int i = c + 1 + lane; i < mk; i += 64) P[q * ps + i] = fma(-ds, P[c * ps + i], P[q * ps + i]);
      if (lane == 0) P[q * ps + c] -= d;
    }
    __syncthreads();
  }
  for (int e = tid; e < 256; e += QT) {
    const int i = e & 15, c = e >> 4;
    if (c < cw && i <= c) it.X[c0 + c + (size_t)n * (c0 + i)] = i < c ? P[c * ps + i] : bet[c];
  }
  __syncthreads();
  for (int c = wv; c < cw; c += QW) {
    double* V = it.A + (size_t)m * (c0 + c);
    for (int i = lane; i < q0; i += 64) V[i] = 0.0;
    for (int i = lane; i < mk; i += 64) {
      const double v = i < c ? 0.0 : (i == c ? 1.0 : scl[c] * P[c * ps + i]);
      P[c * ps + i] = v;
      V[q0 + i] = v;
    }
  }
  __syncthreads();
  {  // V^T V, then T by columns: T(0:c, c) = -tau_c T(0:c, 0:c) V^T v_c
    svd_t4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int base = 4 * wv; base < mk; base += 4 * QW) {
      const double v = base + lg < mk && (!TALL || lr < cw) ? P[lr * ps + base + lg] : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v, v, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) part[wv][(4 * r + lg) * 16 + lr] = acc[r];
    __syncthreads();
    sum_parts(part, w1, tid);
    if (tid < 256) w2[tid] = 0.0;  // T, column-major
    __syncthreads();
    for (int c = 0; c < cw; c++) {
      if (tid < c) {
        double s = 0.0;
        for (int l = tid; l < c; l++) s = fma(w2[tid + 16 * l], w1[16 * l + c], s);
        w2[tid + 16 * c] = -tau[c] * s;
      } else if (tid == c) {
        w2[c + 16 * c] = tau[c];
      }
      __syncthreads();
    }
    if (tid < 256) it.T[256 * k + tid] = w2[tid];
  }
}

// The columns of X and J (n rows each) of a block pair times the 32 x 32 matrix jl
// (row-major, stride 33): strips of 16 rows dealt out to the wavefronts, as the transposed
// product so that loads and stores run along the columns.
__device__ __forceinline__ void times_rotations(double* X, double* J, int n, const double* jl, int p0, int wp, int q0,
                                                int wq, int wv, int lr, int lg) {
  auto valid = [&](int c) { return c < 16 ? c < wp : c - 16 < wq; };
  auto col = [&](int c) { return (size_t)n * (c < 16 ? p0 + c : q0 + c - 16); };
  double a[2][8];
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int s = 0; s < 8; s++) a[t][s] = jl[(4 * s + lg) * 33 + 16 * t + lr];
  const int strips = (n + 15) >> 4;
  for (int st = wv; st < 2 * strips; st += RW) {
    double* M = st < strips ? X : J;
    const int row = 16 * (st < strips ? st : st - strips) + lr;
    double v[8];
#pragma unroll
    for (int s = 0; s < 8; s++) v[s] = (row < n && valid(4 * s + lg)) ? M[row + col(4 * s + lg)] : 0.0;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      svd_t4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 8; s++) d = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][s], v[s], d, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int c = 16 * t + 4 * q + lg;
        if (row < n && valid(c)) M[row + col(c)] = d[q];
      }
    }
  }
}

// The rotation that makes columns of norms^2 al, be and dot product ga orthogonal, as s = sin
// and h = tan of its half angle, or (0, 0) when |ga| <= tol sqrt(al be), tol = sqrt(n) 2^-53
// (the rounding floor of the dot product, the stopping rule of LAPACK's dgesvj), or a norm is
// at most the floor fl (numerically zero); tol2 is tol^2. The angle comes from the hardware's
// approximate reciprocal and roots (2^29 units in the last place: what is left of ga is that much
// smaller, which costs no sweep); s is refined to full precision for the h that came out, so the
// rotation is orthogonal whatever the angle. The sector is of order one and columns below its
// floor stay as they are, so al and be lie between 1e-33 and 1e7 and no product comes near the
// limits of doubles.
struct Rot {
  double s, h;
};
__device__ __forceinline__ Rot rotation(double al, double be, double ga, double tol2, double fl) {
  // cos of twice the angle is |d| / |(d, 2 ga)|; q = cos^2 of the angle
  const double d = be - al, ri = __builtin_amdgcn_rsq(fma(d, d, 4.0 * ga * ga)), q = fma(0.5 * fabs(d), ri, 0.5);
  const double ci = __builtin_amdgcn_rsq(q), c1 = fma(q, ci, 1.0);
  const double h = (d >= 0.0 ? ga : -ga) * ri * ci * __builtin_amdgcn_rcp(c1);
  // 1 / (1 + h^2) = (1 + cos) / 2
  const double w = 0.5 * c1, e = fma(-fma(h, h, 1.0), w, 1.0);
  const bool on = al > fl && be > fl && ga * ga > tol2 * (al * be);
  return on ? Rot{2.0 * h * fma(w, fma(e, e, e), w), h} : Rot{0.0, 0.0};
}
// (u, v) <- (c u - s v, s u + c v), with c = 1 - s h: what rounding and an s that is not quite
// sin take from the columns' orthogonality is smaller than with c by a factor of s, and not of
// one sign (c = 1 / sqrt(1 + t^2) and s = c t round alike over ranges of small angles, and the
// columns' norms drift with every rotation: |U^T U - 1| of 32 x 32 matrices with graded rows and
// columns 6.2e-14 that way, 7.0e-15 this way, of 250 x 240 5.7e-14; the re-joined object's error
// 9.3e-15 and 0.9e-15).
__device__ __forceinline__ void rotate(const Rot& r, double u, double v, double& u1, double& v1) {
  u1 = fma(-r.s, fma(r.h, u, v), u);
  v1 = fma(r.s, fma(-r.h, v, u), v);
}

// Round r of a sweep over the column blocks: workgroup (k, sector) takes block pair k.
// Round 0 rotates every pair of the two blocks' columns, the other rounds the pairs across
// them. A sector whose last sweep rotated nothing is done; one of at most two blocks runs
// all its sweeps in the launch of (0, 0).
__global__ __launch_bounds__(RT) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_svd_round(const DevSvd* __restrict__ jobs, int sweep, int r) {
  __shared__ double part[RW][3][256];
  __shared__ double g[2][32 * 33], jl[32 * 33];
  __shared__ int rotated;
  const DevSvd it = jobs[blockIdx.y];
  const int n = it.n, nb = (n + PB - 1) / PB, nb2 = max(2, nb + (nb & 1)), k = blockIdx.x;
  const bool alone = nb2 == 2;
  if (sweep >= it.max_sweeps || r >= nb2 - 1 || k >= nb2 / 2 || (alone && sweep > 0)) return;
  if (sweep > 0 && it.rot[sweep - 1] == 0) return;
  int bp, bq;
  pair_of(nb2, r, k, bp, bq);
  const int p0 = PB * bp, q0 = PB * bq, wp = min(PB, n - p0), wq = bq < nb ? min(PB, n - q0) : 0;
  if (wq == 0 && r > 0) return;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double fl = it.floor2[0], tol2 = (double)n * (SVD_EPS * SVD_EPS);
  for (;;) {
    {  // Gram matrix: [p p], [p q], [q q] blocks, rows dealt out to the wavefronts
      svd_t4 a0 = {0.0, 0.0, 0.0, 0.0}, a1 = a0, a2 = a0;
      const double* xp = it.X + (size_t)n * (p0 + min(lr, wp - 1));
      const double* xq = it.X + (size_t)n * (wq > 0 ? q0 + min(lr, wq - 1) : p0);
      for (int base = 16 * wv; base < n; base += 16 * RW) {
        double u[4], v[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
          const int row = base + 4 * lg + s;
          u[s] = (row < n && lr < wp) ? xp[row] : 0.0;
          v[s] = (row < n && lr < wq) ? xq[row] : 0.0;
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
          a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s], u[s], a0, 0, 0, 0);
          a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s], v[s], a1, 0, 0, 0);
          a2 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[s], v[s], a2, 0, 0, 0);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int e = (4 * q + lg) * 16 + lr;
        part[wv][0][e] = a0[q];
        part[wv][1][e] = a1[q];
        part[wv][2][e] = a2[q];
      }
    }
    if (tid == 0) rotated = 0;
    __syncthreads();
    for (int e = tid; e < 768; e += RT) {
      const int b = e >> 8, i = (e >> 4) & 15, j = e & 15;
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < RW; w++) s += part[w][b][e & 255];
      if (b == 0) g[0][i * 33 + j] = s;
      else if (b == 2) g[0][(16 + i) * 33 + 16 + j] = s;
      else g[0][i * 33 + 16 + j] = g[0][(16 + j) * 33 + i] = s;
    }
    for (int e = tid; e < 1024; e += RT) jl[(e >> 5) * 33 + (e & 31)] = (e >> 5) == (e & 31) ? 1.0 : 0.0;
    __syncthreads();
    // anything to rotate?
    for (int e = tid; e < 1024; e += RT) {
      const int i = e >> 5, j = e & 31;
      if (i >= j || (r > 0 && (i >= 16 || j < 16))) continue;
      if (rotation(g[0][i * 34], g[0][j * 34], g[0][i * 33 + j], tol2, fl).s != 0.0) rotated = 1;
    }
    __syncthreads();
    if (!rotated) break;
    if (tid == 0 && !alone) atomicAdd(it.rot + sweep, 1);
    // one barrier per round: G is double-buffered and every thread works out the rotations
    // it needs by itself
    const int rounds = r == 0 ? 31 : 16;
    const int pa = (tid >> 4) & 15, pb = tid & 15;  // pairs of this thread's 2 x 2 block of G
    for (int q = 0; q < rounds; q++) {
      const double* gi = g[q & 1];
      double* go = g[(q + 1) & 1];
      auto slots = [&](int a, int& x, int& y) {
        if (r == 0) pair_of(32, q, a, x, y);
        else { x = a; y = 16 + ((a + q) & 15); }
      };
      int u, v;
      slots(pb, u, v);
      const Rot rb = rotation(gi[u * 34], gi[v * 34], gi[u * 33 + v], tol2, fl);
      if (tid < 256) {  // G <- R^T G R, a 2 x 2 block per thread
        int x, y;
        slots(pa, x, y);
        const Rot ra = rotation(gi[x * 34], gi[y * 34], gi[x * 33 + y], tol2, fl);
        double x1, x2, y1, y2;
        rotate(rb, gi[x * 33 + u], gi[x * 33 + v], x1, x2);
        rotate(rb, gi[y * 33 + u], gi[y * 33 + v], y1, y2);
        rotate(ra, x1, y1, go[x * 33 + u], go[y * 33 + u]);
        rotate(ra, x2, y2, go[x * 33 + v], go[y * 33 + v]);
      } else {  // the accumulated rotations' columns u and v, two rows per thread
#pragma unroll
        for (int i = 0; i < 2; i++) {
          double* row = jl + (pa + 16 * i) * 33;
          rotate(rb, row[u], row[v], row[u], row[v]);
        }
      }
      __syncthreads();
    }
    times_rotations(it.X, it.J, n, jl, p0, wp, q0, wq, wv, lr, lg);
    if (!alone) return;
    __syncthreads();
    if (++sweep >= it.max_sweeps) {  // the last sweep allowed rotated
      if (tid == 0) *it.info = 1;
      return;
    }
  }
}

// Singular values of the scaled sector (the norms of X's columns, zero below the floor) in
// falling order and their columns (src).
__global__ __launch_bounds__(JT) void k_svd_sigma(const DevSvd* __restrict__ jobs) {
  __shared__ double sig[SVD_MAXM];
  const DevSvd it = jobs[blockIdx.x];
  const int n = it.n, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const double fl = it.floor2[0];
  for (int j = wv; j < n; j += JW) {
    double s = 0.0;
    for (int i = lane; i < n; i += 64) s = fma(it.X[i + (size_t)n * j], it.X[i + (size_t)n * j], s);
    s = wave_sum(s);
    if (lane == 0) sig[j] = s > fl ? sqrt(s) : 0.0;
  }
  __syncthreads();
  for (int j = tid; j < n; j += JT) {
    int r = 0;
    for (int k = 0; k < n; k++) r += (sig[k] > sig[j] || (sig[k] == sig[j] && k < j)) ? 1 : 0;
    it.src[r] = j;
    it.S[r] = sig[j];
  }
}

// The n-long singular vectors, 16 per workgroup: row perm[i] of vector t is X[i, src[t]] /
// sigma_t (zero for sigma_t = 0), sigma still scaled. VT is written 16 neighbouring t at a time.
__global__ __launch_bounds__(QT) void k_svd_short(const DevSvd* __restrict__ jobs) {
  const DevSvd it = jobs[blockIdx.y];
  const int n = it.n, t0 = PB * blockIdx.x;
  if (t0 >= n) return;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (it.wide) {
    for (int t = t0 + wv; t < min(n, t0 + PB); t += QW) {
      const double sj = it.S[t], inv = sj > 0.0 ? 1.0 / sj : 0.0;
      const double* x = it.X + (size_t)n * it.src[t];
      for (int i = lane; i < n; i += 64) it.U[it.perm[i] + (size_t)n * t] = x[i] * inv;
    }
    return;
  }
  const int t = t0 + (threadIdx.x & 15);
  if (t >= n) return;
  const double sj = it.S[t], inv = sj > 0.0 ? 1.0 / sj : 0.0;
  const double* x = it.X + (size_t)n * it.src[t];
  for (int i = threadIdx.x >> 4; i < n; i += QT / 16) it.VT[t + (size_t)n * it.perm[i]] = x[i] * inv;
}

// The m-long singular vectors Q J, 16 of them per workgroup: the columns src[t] of J padded
// to m rows (or, to complete a basis, the unit vectors e_t), in LDS, through the panels'
// reflectors in falling order (I - V T V^T). complete: only the vectors with sigma_t = 0; else the
// singular values also lose their scale. TALL (as in k_qr_step): the vectors in their columns
// of W, which the factorisation left free, instead of LDS.
template <bool TALL>
__global__ __launch_bounds__(QT) void k_svd_long(const DevSvd* __restrict__ jobs, int complete) {
  extern __shared__ double panel[];
  __shared__ double part[QW][256];
  __shared__ double w1[256], w2[256];
  const DevSvd it = jobs[blockIdx.y];
  const int m = it.m, n = it.n, nb = (n + PB - 1) / PB, t0 = PB * blockIdx.x;
  if (t0 >= n || (m > SVD_MAXM) != TALL) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, lr = lane & 15, lg = lane >> 4;
  const int tw = TALL ? min(PB, n - t0) : PB;  // columns of P
  double* P;                                   // 16 columns of m
  if constexpr (TALL) P = it.W + (size_t)m * t0;
  else P = panel;
  if (!complete && tid < PB && t0 + tid < n && it.floor2[1] > 0.0) it.S[t0 + tid] *= 1.0 / it.floor2[1];
  for (int c = wv; c < tw; c += QW) {
    const int t = t0 + c;
    const double* x = it.J + (t < n && !complete ? (size_t)n * it.src[t] : 0);
    for (int i = lane; i < m; i += 64)
      P[c * m + i] = t >= n ? 0.0 : complete ? (i == t ? 1.0 : 0.0) : (i < n ? x[i] : 0.0);
  }
  __syncthreads();
  for (int k = nb - 1; k >= 0; k--) {
    const int r0 = PB * k, cw = min(PB, n - r0);
    const double* V = it.A + (size_t)m * r0;
    const double* T = it.T + 256 * k;
    svd_t4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int base = r0 + 16 * wv; base < m; base += 16 * QW) {
      double v[4], c[4];
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int row = base + 4 * lg + s;
        v[s] = (row < m && lr < cw) ? V[row + (size_t)m * lr] : 0.0;
        c[s] = (row < m && lr < tw) ? P[lr * m + row] : 0.0;
      }
#pragma unroll
      for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v[s], c[s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) part[wv][(4 * r + lg) * 16 + lr] = acc[r];
    __syncthreads();
    sum_parts(part, w1, tid);
    __syncthreads();
    if (tid < 256) {
      const int i = tid >> 4, q = tid & 15;
      double s = 0.0;
      for (int l = i; l < cw; l++) s = fma(T[i + 16 * l], w1[16 * l + q], s);
      w2[tid] = s;
    }
    __syncthreads();
    for (int base = r0 + 16 * wv; base < m; base += 16 * QW) {
      const int row = base + lr;
      svd_t4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const double v = (row < m && 4 * s + lg < cw) ? V[row + (size_t)m * (4 * s + lg)] : 0.0;
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(w2[16 * (4 * s + lg) + lr], v, d, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (row < m && 4 * r + lg < tw) P[(4 * r + lg) * m + row] -= d[r];
    }
    __syncthreads();
  }
  if (it.wide) {  // 16 neighbouring t at a time
    const int t = t0 + (tid & 15);
    if (t >= n || (complete && it.S[t] > 0.0)) return;
    for (int i = tid >> 4; i < m; i += QT / 16) it.VT[t + (size_t)n * i] = P[(tid & 15) * m + i];
    return;
  }
  for (int c = wv; c < PB; c += QW) {
    const int t = t0 + c;
    if (t >= n || (complete && it.S[t] > 0.0)) continue;
    for (int i = lane; i < m; i += 64) it.U[i + (size_t)m * t] = P[c * m + i];
  }
}

// For a basis to complete (n x n; U with leading dimension n, or VT's rows): W = the vectors
// with sigma_t > 0 in order, zeros for the rest.
__global__ __launch_bounds__(JT) void k_svd_gather(const DevSvd* __restrict__ jobs) {
  const DevSvd it = jobs[blockIdx.x];
  const int n = it.n;
  for (int e = threadIdx.x; e < n * n; e += JT) {
    const int i = e % n, t = e / n;
    it.W[e] = it.S[t] > 0.0 ? (it.wide ? it.VT[t + (size_t)n * i] : it.U[i + (size_t)n * t]) : 0.0;
  }
}

size_t qr_lds(int m) { return (size_t)PB * m * sizeof(double); }

// the LDS of the QR kernels
void svd_setup() {
  hip_check(hipFuncSetAttribute((const void*)k_qr_step<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)qr_lds(SVD_MAXM)), "SVD kernel LDS");
  hip_check(hipFuncSetAttribute((const void*)k_svd_long<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)qr_lds(SVD_MAXM)), "SVD kernel LDS");
}

// panels of the widest sector, rows of the longest with its panel in LDS (0: none), any longer
struct Extent {
  int nb = 0, m = 0;
  bool tall = false;
  explicit Extent(const std::vector<DevSvd>& jobs) {
    for (const DevSvd& j : jobs) {
      nb = std::max(nb, (j.n + PB - 1) / PB);
      if (j.m > SVD_MAXM) tall = true;
      else m = std::max(m, j.m);
    }
  }
};

void launch_qr(const DevSvd* d, const std::vector<DevSvd>& jobs, hipStream_t s) {
  const Extent x(jobs);
  for (int k = 0; k < x.nb; k++) {
    const dim3 grid(x.nb - k, (int)jobs.size());
    if (x.m > 0) hipLaunchKernelGGL(k_qr_step<false>, grid, dim3(QT), qr_lds(x.m), s, d, k);
    if (x.tall) hipLaunchKernelGGL(k_qr_step<true>, grid, dim3(QT), 0, s, d, k);
  }
}

void launch_long(const DevSvd* d, const std::vector<DevSvd>& jobs, int complete, hipStream_t s) {
  const Extent x(jobs);
  const dim3 grid(x.nb, (int)jobs.size());
  if (x.m > 0) hipLaunchKernelGGL(k_svd_long<false>, grid, dim3(QT), qr_lds(x.m), s, d, complete);
  if (x.tall) hipLaunchKernelGGL(k_svd_long<true>, grid, dim3(QT), 0, s, d, complete);
}

}  // namespace

void svd_batch(std::vector<DevSvd>& jobs, DBuf<DevSvd>& buf, int* h_rot, const int* d_rot, hipStream_t s) {
  if (jobs.empty()) return;
  svd_setup();
  // widest first: their workgroups set a launch's time and start first
  std::stable_sort(jobs.begin(), jobs.end(), [](const DevSvd& a, const DevSvd& b) { return a.n > b.n; });
  buf.upload(jobs, s);
  const int nj = (int)jobs.size();
  hipLaunchKernelGGL(k_svd_sort, dim3(nj), dim3(JT), 0, s, buf.p);
  hipLaunchKernelGGL(k_svd_copy, dim3(SVD_CHUNKS, nj), dim3(QT), 0, s, buf.p);
  launch_qr(buf.p, jobs, s);
  // The first launch takes every sector; the next ones those of more than two blocks. The
  // counters are looked at from the fifth sweep on: none ends before it.
  const int nb = (jobs[0].n + PB - 1) / PB, nb2 = std::max(2, nb + (nb & 1)), most = jobs[0].max_sweeps;
  int nl = 0;
  while (nl < nj && jobs[nl].n > SVD_ALONE) nl++;
  for (int sweep = 0; sweep < (nl > 0 ? most : 1); sweep++) {
    for (int r = 0; r < nb2 - 1; r++)
      hipLaunchKernelGGL(k_svd_round, dim3(nb2 / 2, sweep == 0 && r == 0 ? nj : nl), dim3(RT), 0, s, buf.p, sweep, r);
    if (nl == 0 || sweep + 1 < std::min(5, most)) continue;
    hip_check(hipMemcpyAsync(h_rot, d_rot, (size_t)nj * SVD_SWEEPS * sizeof(int), hipMemcpyDeviceToHost, s), "SVD counters");
    hip_check(hipStreamSynchronize(s), "SVD sweeps");
    bool any = false;
    for (int q = 0; q < nl; q++) any |= h_rot[(jobs[q].rot - d_rot) + sweep] != 0;
    if (!any) break;
  }
  hipLaunchKernelGGL(k_svd_sigma, dim3(nj), dim3(JT), 0, s, buf.p);
  hipLaunchKernelGGL(k_svd_short, dim3(nb, nj), dim3(QT), 0, s, buf.p);
  launch_long(buf.p, jobs, 0, s);
  hip_check(hipGetLastError(), "SVD kernels");
}

void svd_complete(std::vector<DevSvd>& jobs, DBuf<DevSvd>& buf, hipStream_t s) {
  if (jobs.empty()) return;
  for (DevSvd& j : jobs) {  // the n-long side becomes the "long" one of an n x n problem
    j.m = j.n;
    j.wide = !j.wide;
  }
  buf.upload(jobs, s);
  hipLaunchKernelGGL(k_svd_gather, dim3((int)jobs.size()), dim3(JT), 0, s, buf.p);
  launch_qr(buf.p, jobs, s);
  launch_long(buf.p, jobs, 1, s);
  hip_check(hipGetLastError(), "SVD completion");
}

}  // namespace chm
