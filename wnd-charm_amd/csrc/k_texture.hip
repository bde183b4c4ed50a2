// Texture feature kernels: Haralick (co-occurrence statistics f1..f14),
// Tamura, Comb moments and Radon.  FP64.
//
// Haralick f14 needs the eigenvalue at index 2 of the real Schur form that
// the reference's Eigen 3.1.2 EigenSolver produces (CVIPtexture.cpp:993-1023),
// so Q, the Householder Hessenberg reduction and the Francis double-shift QR
// below perform the same floating-point operations in the same order as the
// CPU oracle's restatement of that algorithm: every reduction that feeds a
// decision is a per-thread sequential loop, parallelism is across the
// independent rows / columns a reflector touches.
#include <utility>
#include "common.hpp"
#include "kernels.hpp"
#include "schur_math.hpp"

namespace wnd {

// Memory fence for lanes of one wavefront exchanging values through LDS:
// a wave's LDS operations execute in issue order, so only compiler
// reordering has to be prevented.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- Eigen 3.1.2 evaluation orders (SSE2, two doubles per packet) used by
// the reference's f14 on row-major arrays (CVIPtexture.cpp:961-1023):
// eigen_redux is DenseBase::sum() over a contiguous range with linear
// vectorized traversal (Core/Redux.h:193-248); s is the index of the first
// 16-byte-aligned term.  x(k) supplies term k.
template <class F>
__device__ __forceinline__ double eigen_redux(int m, int s, F x) {
  if (s > m) s = m;
  const int as = ((m - s) / 2) * 2, as2 = ((m - s) / 4) * 4;
  const int end = s + as, end2 = s + as2;
  double res;
  if (as) {
    double a0 = x(s), a1 = x(s + 1);
    if (as > 2) {
      double b0 = x(s + 2), b1 = x(s + 3);
      for (int k = s + 4; k < end2; k += 4) {
        a0 = a0 + x(k); a1 = a1 + x(k + 1);
        b0 = b0 + x(k + 2); b1 = b1 + x(k + 3);
      }
      a0 = a0 + b0; a1 = a1 + b1;
      if (end > end2) { a0 = a0 + x(end2); a1 = a1 + x(end2 + 1); }
    }
    res = a0 + a1;
    for (int k = 0; k < s; k++) res = res + x(k);
    for (int k = end; k < m; k++) res = res + x(k);
  } else {
    res = x(0);
    for (int k = 1; k < m; k++) res = res + x(k);
  }
  return res;
}

// ===================================================================== Haralick
// quantisation (haralick.cpp:29-37) and tone presence
__global__ void k_har_quant(const Img *imgs, const Stats *st, const HarDesc *hd) {
  const Img im = imgs[blockIdx.y];
  const HarDesc H = hd[blockIdx.y];
  const Stats S = st[blockIdx.y];
  const long n = (long)im.h * im.w;
  const double scale255 = (255.0 / (S.mx - S.mn));
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const double t = (im.p[i] - S.mn) * scale255;
    const int g = (t >= 0 && t < 256) ? (int)t : (t >= 256 ? 255 : 0);
    H.gray[i] = (uint8_t)g;
    H.lut[g] = 1;  // benign race: every writer stores 1
  }
}

// tone LUT (CVIPtexture.cpp:400-414): rank of each present gray level
__global__ void k_har_lut(const HarDesc *hd) {
  const HarDesc H = hd[blockIdx.x];
  if (threadIdx.x == 0) {
    int it = 0;
    for (int g = 0; g < 256; g++) H.lut[g] = H.lut[g] ? it++ : -1;
    *H.ng = it;
  }
}

// co-occurrence counts (CoOcMat_Angle_*, CVIPtexture.cpp:455-614) in LDS as the
// upper triangle of the symmetric matrix, then P = count / total
__device__ __forceinline__ int tri(int i, int j) { return i * (2 * 256 - i + 1) / 2 + (j - i); }

__global__ void __launch_bounds__(1024) k_har_cooc(const Img *imgs, const HarDesc *hd) {
  extern __shared__ uint32_t cnt[];  // 256*257/2
  __shared__ int lut[256];
  __shared__ int total;
  const int angle = blockIdx.x;
  const Img im = imgs[blockIdx.y];
  const HarDesc H = hd[blockIdx.y];
  const int ng = *H.ng;
  for (int e = threadIdx.x; e < 256 * 257 / 2; e += blockDim.x) cnt[e] = 0;
  if (threadIdx.x < 256) lut[threadIdx.x] = H.lut[threadIdx.x];
  if (threadIdx.x == 0) total = 0;
  __syncthreads();
  const int rows = im.h, cols = im.w;
  const int n = rows * cols;  // planes hold fewer than 2^31 pixels: 32-bit index arithmetic
  const gptr<const uint8_t> gray = to_global((const uint8_t *)H.gray);
  int local = 0;
  // four pixels per thread and pass: the pixel and neighbour loads are clamped
  // into the plane and issued together, the pairs outside it are not counted
  for (int i0 = threadIdx.x; i0 < n; i0 += 4 * blockDim.x) {
    int gv[4], g2v[4];
    bool okv[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int i = i0 + u * (int)blockDim.x;
      bool ok = i < n;
      const int ii = ok ? i : 0;
      const int row = ii / cols, col = ii - row * cols;
      int r2 = row, c2 = col;
      if (angle == 0) { c2 = col + 1; ok = ok && c2 < cols; }
      else if (angle == 1) { r2 = row + 1; c2 = col - 1; ok = ok && r2 < rows && c2 >= 0; }
      else if (angle == 2) { r2 = row + 1; ok = ok && r2 < rows; }
      else { r2 = row + 1; c2 = col + 1; ok = ok && r2 < rows && c2 < cols; }
      gv[u] = gray[ii];
      g2v[u] = gray[ok ? r2 * cols + c2 : ii];
      okv[u] = ok;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (!okv[u] || !gv[u] || !g2v[u]) continue;
      const int x = lut[gv[u]], y = lut[g2v[u]];
      if (x == y) atomicAdd(&cnt[tri(x, x)], 2u);
      else atomicAdd(&cnt[x < y ? tri(x, y) : tri(y, x)], 1u);
      local += 2;
    }
  }
  atomicAdd(&total, local);
  __syncthreads();
  const int count = total;
  double *P = H.P + (long)angle * ng * ng;
  for (int e = threadIdx.x; e < ng * ng; e += blockDim.x) {
    const int i = e / ng, j = e - i * ng;
    const uint32_t c = cnt[i <= j ? tri(i, j) : tri(j, i)];
    P[e] = count == 0 ? 0.0 : (double)c / count;
  }
  if (threadIdx.x == 0) H.count[angle] = count;
}

// f1..f13 (CVIPtexture.cpp:631-958) and Q (_Q_calc_eigen, 961-987) per angle
__global__ void __launch_bounds__(256) k_har_stats(const HarDesc *hd) {
  __shared__ double px[256], py[256], pxpy_s[512], pxpy_d[256];
  __shared__ double lse[512], lde[256], lhx[256], lhy[256];  // the entropy terms, formed in parallel
  __shared__ double shd[4];
  const int angle = blockIdx.x;
  const HarDesc H = hd[blockIdx.y];
  const int ng = *H.ng;
  const gptr<const double> P = to_global((const double *)H.P + (long)angle * ng * ng);
  const int t = threadIdx.x;
  const double LOG2 = log10(2.0), EPS = 0.000000001;
  // exact per-row / per-column marginals (sequential, as the reference
  // loops).  P is symmetric (k_har_cooc stores the counts as a triangle),
  // so row t equals column t term by term and both sums walk the column,
  // which the lanes read coalesced.
  // (each sequential sum loads its terms eight at a time, then adds them in
  // order: the loads are in flight together instead of one latency a term)
  if (t < ng) {
    double b = 0;
    int i = 0;
    for (; i + 8 <= ng; i += 8) {
      double v[8];
#pragma unroll
      for (int q = 0; q < 8; q++) v[q] = P[(i + q) * ng + t];
#pragma unroll
      for (int q = 0; q < 8; q++) b += v[q];
    }
    for (; i < ng; i++) b += P[i * ng + t];
    px[t] = b;
    py[t] = b;
  }
  // Pxpy[i+j] (anti-diagonals, raster order) and Pxpy[|i-j|] (f2, f10, f11)
  for (int k = t; k < 2 * ng - 1; k += blockDim.x) {
    double s = 0;
    const int i0 = k - (ng - 1) > 0 ? k - (ng - 1) : 0, i1 = k < ng - 1 ? k : ng - 1;
    int i = i0;
    for (; i + 8 <= i1 + 1; i += 8) {
      double v[8];
#pragma unroll
      for (int q = 0; q < 8; q++) v[q] = P[(i + q) * ng + (k - i - q)];
#pragma unroll
      for (int q = 0; q < 8; q++) s += v[q];
    }
    for (; i <= i1; i++) s += P[i * ng + (k - i)];
    pxpy_s[k] = s;
  }
  if (t < ng) {
    // both loads at clamped (in-range) columns every row, so they are not
    // behind a branch and can be in flight together; the adds are as before
    double s = 0;
    int i = 0;
    for (; i + 4 <= ng; i += 4) {
      double lo[4], hi[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        lo[q] = P[(i + q) * ng + max(i + q - t, 0)];
        hi[q] = P[(i + q) * ng + min(i + q + t, ng - 1)];
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (i + q - t >= 0) s += lo[q];
        if (t > 0 && i + q + t < ng) s += hi[q];
      }
    }
    for (; i < ng; i++) {
      const double lo = P[i * ng + max(i - t, 0)], hi = P[i * ng + min(i + t, ng - 1)];
      if (i - t >= 0) s += lo;
      if (t > 0 && i + t < ng) s += hi;
    }
    pxpy_d[t] = s;
  }
  __syncthreads();
  // raster double sums (parallel)
  double f1 = 0, tmp3 = 0, mean4 = 0, idm = 0, ent = 0, hxy1 = 0, hxy2 = 0;
  const int nn = ng * ng, bs = blockDim.x;
  double pb[4] = {0.0, 0.0, 0.0, 0.0};  // this thread's next four elements, loaded ahead
  if (nn > 0)
#pragma unroll
    for (int q = 0; q < 4; q++) pb[q] = P[min(t + q * bs, nn - 1)];
  for (int e = t; e < nn; e += bs) {
    const int i = e / ng, j = e - i * ng;
    const double p = pb[0];
    pb[0] = pb[1];
    pb[1] = pb[2];
    pb[2] = pb[3];
    pb[3] = P[min(e + 4 * bs, nn - 1)];  // four elements ahead (clamped: unused past the end)
    f1 += p * p;
    tmp3 += i * j * p;
    mean4 += i * p;
    idm += p / (1 + (i - j) * (i - j));
    ent += p * log10(p + EPS) / LOG2;
    const double lg = log10(px[i] * py[j] + EPS);
    hxy1 -= p * lg / LOG2;
    hxy2 -= px[i] * py[j] * lg / LOG2;
  }
  f1 = block_reduce(f1, SumOp(), shd);
  tmp3 = block_reduce(tmp3, SumOp(), shd);
  mean4 = block_reduce(mean4, SumOp(), shd);
  idm = block_reduce(idm, SumOp(), shd);
  ent = block_reduce(ent, SumOp(), shd);
  hxy1 = block_reduce(hxy1, SumOp(), shd);
  hxy2 = block_reduce(hxy2, SumOp(), shd);
  double var4 = 0;
  {
    int e = t;
    for (; e + 7 * bs < nn; e += 8 * bs) {
      double v[8];
#pragma unroll
      for (int q = 0; q < 8; q++) v[q] = P[e + q * bs];
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int i = (e + q * bs) / ng;
        var4 += (i - mean4) * (i - mean4) * v[q];
      }
    }
    for (; e < nn; e += bs) {
      const int i = e / ng;
      var4 += (i - mean4) * (i - mean4) * P[e];
    }
  }
  var4 = block_reduce(var4, SumOp(), shd);
  // the terms of the sum entropy, difference entropy and HX / HY, each formed
  // by one thread with the serial loop's operations; thread 0 then adds them
  // in the loops' order
  for (int k = t; k <= 2 * ng - 2; k += blockDim.x) {
    const double v = pxpy_s[k];
    lse[k] = v * log10(v + EPS) / LOG2;
  }
  if (t < ng) {
    lde[t] = pxpy_d[t] * log10(pxpy_d[t] + EPS) / LOG2;
    lhx[t] = px[t] * log10(px[t] + EPS) / LOG2;
    lhy[t] = py[t] * log10(py[t] + EPS) / LOG2;
  }
  __syncthreads();
  if (t == 0) {
    double *F = H.feat + angle * 14;
    F[0] = f1;
    double bigsum = 0;
    for (int n = 0; n < ng; n++) bigsum += n * n * pxpy_d[n];
    F[1] = bigsum;
    double meanx = 0, sum_sqrx = 0;
    for (int i = 0; i < ng; i++) { meanx += px[i] * i; sum_sqrx += px[i] * i * i; }
    const double sd = sqrt(sum_sqrx - (meanx * meanx));
    F[2] = (sd * sd == 0) ? 1.0 : (tmp3 - meanx * meanx) / (sd * sd);
    F[3] = var4;
    F[4] = idm;
    double savg = 0;
    for (int i = 0; i <= 2 * ng - 2; i++) savg += i * pxpy_s[i];
    F[5] = savg;
    double se = 0;
    for (int i = 2; i <= 2 * ng; i++) se -= lse[i - 2];  // i - 2 <= 2 ng - 2 throughout
    F[7] = se;
    double sv = 0;
    for (int i = 0; i <= 2 * ng - 2; i++) sv += (i - se) * (i - se) * pxpy_s[i];
    F[6] = sv;
    F[8] = -ent;
    double s = 0, ss = 0, de = 0;
    for (int i = 0; i < ng; i++) { s += i * pxpy_d[i]; ss += i * i * pxpy_d[i]; }
    F[9] = ss - s * s;
    for (int i = 0; i < ng; i++) de += lde[i];
    F[10] = -de;
    double hx = 0, hy = 0;
    for (int i = 0; i < ng; i++) {
      hx -= lhx[i];
      hy -= lhy[i];
    }
    const double hxy = -ent;
    const double mxh = hx > hy ? hx : hy;
    F[11] = (mxh == 0) ? 1.0 : (hxy - hxy1) / mxh;
    F[12] = sqrt(fabs(1 - exp(-2.0 * (hxy2 - hxy))));
  }
  // marginals of _Q_calc_eigen: px = P.rowwise().sum() (row t of the
  // row-major array starts at linear index t*ng; its terms are read down
  // column t, equal by symmetry), py = P.colwise().sum() (strided: a
  // running sum, equal to py above)
  if (t < ng) {
    H.marg[angle * 512 + t] = eigen_redux(ng, (int)(((long)t * ng) & 1), [&](int k) { return P[(long)k * ng + t]; });
    H.marg[angle * 512 + 256 + t] = py[t];
  }
}

// Q (_Q_calc_eigen, CVIPtexture.cpp:961-987):
//   Q(i,j) = (P.row(i)*P.row(j) / (px(i) py + 1e-13)).sum(),
// an Eigen redux over an aligned expression: terms k < 4*floor(Ng/4) go to
// four accumulators by k mod 4, which are paired (0+2, 1+3); the next two
// terms (if Ng mod 4 >= 2) join the pairs, the pairs are added, and an odd
// last term comes last.  Every term is >= +0, so an accumulator that
// starts at +0 and skips zero terms holds the same bits: each row visits
// only the k with P(i,k) != 0 (compacted per wavefront), and skips
// P(j,k) == 0.  P is symmetric (pairs are counted both ways), so P(j,k) is
// read as P(k,j): along row k, coalesced over j.
constexpr int QRB = 4;  // row blocks per angle
struct Redux4 {
  double a0, a1, a2, a3, e0, e1, tl;
};
// k is the same for every lane of a wavefront, so the branches are uniform
__device__ __forceinline__ void r4_add(Redux4 &r, int k, int as2, int as, double term) {
  if (k < as2 || (as2 == 0 && k < as)) {  // four accumulators; ng 2..3: the single packet (x0, x1)
    switch (k & 3) {
      case 0: r.a0 += term; break;
      case 1: r.a1 += term; break;
      case 2: r.a2 += term; break;
      default: r.a3 += term; break;
    }
  } else if (k < as) {
    if (k == as2) r.e0 += term;
    else r.e1 += term;
  } else {
    r.tl += term;  // odd last term (or x0 when ng == 1)
  }
}
__device__ __forceinline__ double r4_finish(const Redux4 &r, int ng) {
  if (ng == 1) return r.tl;
  double res;
  if (ng >= 4) {
    double l0 = r.a0 + r.a2, l1 = r.a1 + r.a3;
    if ((ng / 2) * 2 > (ng / 4) * 4) { l0 = l0 + r.e0; l1 = l1 + r.e1; }
    res = l0 + l1;
  } else {
    res = r.a0 + r.a1;
  }
  if (ng & 1) res = res + r.tl;
  return res;
}

__global__ void __launch_bounds__(256) k_har_q(const HarDesc *hd, int nimg) {
  __shared__ int lk[4][256];
  __shared__ double la[4][256], ld[4][256];
  int item, rb;
  if (!xcd_item(QRB, 4 * nimg, item, rb)) return;  // the row blocks of one P share an XCD
  const int angle = item & 3;
  const HarDesc H = hd[item >> 2];
  const int ng = *H.ng;
  const double *P = H.P + (long)angle * ng * ng;
  const double *px = H.marg + angle * 512, *py = px + 256;
  double *Q = H.Q + (long)angle * ng * ng;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int i = rb * 4 + w; i < ng; i += QRB * 4) {
    const double pxi = px[i];
    int cnt = 0;
    for (int k0 = 0; k0 < ng; k0 += 64) {
      const int k = k0 + lane;
      const double a = k < ng ? to_global(P)[(long)i * ng + k] : 0.0;
      const unsigned long long m = __ballot(a != 0.0);
      if (a != 0.0) {
        const int pos = cnt + __popcll(m & ((1ull << lane) - 1));
        lk[w][pos] = k;
        la[w][pos] = a;
        ld[w][pos] = py[k] * pxi + 0.0000000000001;
      }
      cnt += __popcll(m);
    }
    wave_sync();
    // four output columns per lane, one pass over the row's list
    const int as2 = (ng / 4) * 4, as = (ng / 2) * 2;
    Redux4 r[4];
#pragma unroll
    for (int q = 0; q < 4; q++) r[q] = Redux4{0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    // list entries in order, two at a time so that 8 row loads are in flight
    const gptr<const double> Pg = to_global(P);
    int kk = 0;
    for (; kk + 2 <= cnt; kk += 2) {
      int k[2];
      double a[2], d[2], b[2][4];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        k[u] = lk[w][kk + u];
        a[u] = la[w][kk + u];
        d[u] = ld[w][kk + u];
      }
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int col = lane + 64 * q;
          const double v = Pg[(unsigned)(k[u] * ng + min(col, ng - 1))];
          b[u][q] = col < ng ? v : 0.0;
        }
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (b[u][q] != 0.0) r4_add(r[q], k[u], as2, as, (a[u] * b[u][q]) / d[u]);
    }
    for (; kk < cnt; kk++) {
      const int k = lk[w][kk];
      const double a = la[w][kk], d = ld[w][kk];
      double b[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int col = lane + 64 * q;
        const double v = Pg[(unsigned)(k * ng + min(col, ng - 1))];
        b[q] = col < ng ? v : 0.0;
      }
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (b[q] != 0.0) r4_add(r[q], k, as2, as, (a * b[q]) / d);
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (lane + 64 * q < ng) Q[(long)i * ng + lane + 64 * q] = r4_finish(r[q], ng);
    wave_sync();  // the lists are rebuilt for the next row
  }
}

// --------------------------------------------------------- eigenvalues of Q
// Householder vector (Eigen makeHouseholder) of x[0..m-1], one thread.
__device__ void make_hh(const double *x, int m, double *ess, double *tau, double *beta) {
  double tail = 0;
  for (int i = 1; i < m; i++) tail += x[i] * x[i];
  const double c0 = x[0];
  if (tail == 0.0) {
    *tau = 0; *beta = c0;
    for (int i = 1; i < m; i++) ess[i - 1] = 0;
    return;
  }
  double b = sqrt(c0 * c0 + tail);
  if (c0 >= 0) b = -b;
  for (int i = 1; i < m; i++) ess[i - 1] = x[i] / (c0 - b);
  *tau = (b - c0) / b;
  *beta = b;
}

// One block per (angle, image): Hessenberg reduction of Q (n x n, row-major,
// in place), then (k_har_qr) the Francis QR on the active windows.  Only the
// values of index 0..2 of the Schur diagonal are consumed (f14 = sqrt of
// index 2 when that eigenvalue is real).
constexpr int QB = 28;       // bulge-chase steps per LDS window
constexpr int QW = QB + 4;   // window side (<= 64: one wavefront lane per row/column)
constexpr int QWP = QW + 1;  // padded LDS row of the window
// window and strip tiles are loaded as two rows of 32 lanes per wave instruction
static_assert(QW <= 32 && QW % 2 == 0 && QB + 2 <= QW, "QR window tiles must fit 32-lane rows");
static_assert(QW * QWP >= 256, "the window buffer also holds the n <= 256 row sums of the Schur norm");
// The value of the neighbouring lane (lane ^ 1).
__device__ __forceinline__ double lane_xor1(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_mov_dpp((int)b, 0xB1, 0xf, 0xf, true);  // quad_perm 1,0,3,2
  const unsigned hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xB1, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | lo);
}

constexpr int HT8 = 9;          // padded row of a wave's 32 x 8 staging tile
constexpr int HTW = 32 * HT8;   // a wave's tile
constexpr int HCAP = 16384;     // doubles of the matrix kept in LDS
// k_har_hess takes a CU per matrix.  Where HESS_MANY entries or more have at most
// HESS_SMALL tones, a launch of one wave and 12 KB of LDS per matrix takes those:
// 4,000 matrices of 4 tones 72 us (164 by whole CUs, 132 before there were such),
// of 16 252 (773, 903), of 32 565 (1796, 2133).  It would follow the large ones'
// launch, though, and fewer small matrices run beside those for nothing.
constexpr int HESS_SMALL = 32, HESS_MANY = 256;
// all waves' LDS accesses complete; global stores may be in flight
__device__ __forceinline__ void lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One block per (angle, image): HessenbergDecomposition::_compute
// (Eigenvalues/HessenbergDecomposition.h:292-318) of Q (n x n, row-major, in
// place).  Rows 0..i only ever receive the right reflectors of steps >= i,
// and nothing else reads them, so step i works on the active rows and columns
// i+1..n-1 and the rows above are brought up to date by k_har_hess_rows; every element still receives the same operations in the same order.
// Two passes over the active block per step:
//   row pass     A = H A of step i (row i+1 -= tau*tw, the rows below -=
//                (tau*ess)*tw; tw = the left dot of the column pass before),
//                then the row dots in Eigen's RowMajor GEMV order
//                (general_matrix_vector_product<RowMajor>,
//                GeneralMatrixVector.h:289-552): even and odd terms in two
//                lanes, the lanes added, an odd last term, + A(r, i+1).  The
//                two lanes are two threads: 32 rows per wave.
//   column i+1   A = A H on column i+1 (factor 1), then the reflector of step
//                i+1 from it (kept in the co-occurrence buffer, free once Q is
//                built, for k_har_hess_rows).
//   column pass  A = A H on columns i+2..n-1 and the left dot of step i+1 on
//                them, in Eigen's ColMajor GEMV order on bottom^T
//                (general_matrix_vector_product<ColMajor>,
//                GeneralMatrixVector.h:31-285): inner terms (rows i+3..n-1) in
//                groups of four (g, g+o1, g+2, g+o3), added pairwise for
//                outputs in the packet range and left to right for an odd last
//                output; leftover terms one by one; a skipped leading term
//                last; then + A(i+2, c).  Two threads per column take two rows
//                of each group.
// The last K columns of the active rows live in LDS (K = 64, 96, then all 128
// once 128 rows are left); the columns before them are streamed from global
// memory, the row pass through a wave-private tile with the next 32 columns in
// flight.  Column c of resident row r lies at c ^ (r & 31) within its 32, so
// that neither walking rows nor walking columns conflicts.
//
// What bounds it: per step the latency of the two passes over the streamed
// columns (15,000 and 19,000 cycles at 190 rows) and four barriers; with all
// columns resident a step takes 13,000 cycles, its serial dots, the reflector's
// norm and LDS round trips.  The kernel before, 256 threads with every column
// streamed and the rows above updated by the same block, took 8.5 ms for one
// 256 x 256 image's 48 matrices, now 3.3 with k_har_hess_rows, and 167 ms for
// 19,200 (0.77 TB at the fabric's 4.6 TB/s), now 132.
// Eigen's last step (one row below the diagonal) scales by 1 - tau with
// tau = 0 (a one-element reflector): an exact no-op, not performed.
template <int NW, int NMAX>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, NW == 1 ? 4 : 2)))
k_har_hess(const HarDesc *hd, const int *order) {
  constexpr bool SMALL = NMAX <= 32;    // every column resident, rows and columns of one wave
  __shared__ double res[SMALL ? NMAX * 32 : HCAP];  // resident columns
  __shared__ __align__(16) double tile[NW * HTW];  // per wave: staging; then the squares of its rows' x
  __shared__ __align__(16) double2 twe[NMAX];      // by column: left dot, essential element of step i
  __shared__ __align__(16) double2 tun[NMAX];      // by row: tau * right dot of step i, essential of step i (row pass) / i+1 (column pass)
  __shared__ double lf[NMAX];            // by row: left factor of step i
  __shared__ double xc[NMAX];            // by row: column i+1 after step i
  __shared__ double sc[4];
  // entries by decreasing n: the large ones, the small ones, those of n < 3 (Hessenberg as they are)
  const int e = blockIdx.y, first = SMALL ? order[gridDim.y + ORDER_LARGE] : 0;
  if (e < first || e >= order[gridDim.y + (SMALL ? ORDER_END : ORDER_LARGE)]) return;
  const int angle = blockIdx.x;
  const HarDesc H = hd[order[blockIdx.y]];
  const int n = __builtin_amdgcn_readfirstlane(*H.ng);
  gptr<double> A = to_global(H.Q + (long)angle * n * n);
  gptr<double> Rf = to_global(H.P + (long)angle * n * n);  // reflector store
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool odd_n = n & 1;
  int K = 0, cK = n, r0 = 0;  // resident: columns cK.., rows r0.. (row r at (r - r0) * K)
#define AT(r, c) A[(unsigned)((r) * n + (c))]
#define RES(r, c) res[((r) - r0) * K + (((c) - cK) ^ ((r) & 31))]

  // Reflector of column s below the diagonal (Eigen makeHouseholderInPlace)
  // from xc[s+1..n-1] and the squares of xc (row base + k at tile row k): the
  // column is strided in row-major storage, so Eigen sums the tail in order.
  // Writes beta and the zeros of the Hessenberg form into column s, the
  // reflector into row s of Rf (essential part, tau in column n-1) and tun.y.
  auto reflector = [&](int s, int base) {
    if (wave == 0) {
      const double c0 = xc[s + 1];
      double tail = 0;
      for (int w = 0; w * 32 < n - base; w++) {
        const int k0 = s + 2 - base - 32 * w, k1 = min(32, n - base - 32 * w);  // tile rows k0..k1-1 of this wave
        const double2 *q = (const double2 *)(tile + w * HTW);
        double2 v[16];
#pragma unroll
        for (int k = 0; k < 16; k++) v[k] = q[k];
        if (k0 <= 0 && k1 == 32) {
#pragma unroll
          for (int k = 0; k < 16; k++) {
            tail += v[k].x;
            tail += v[k].y;
          }
        } else {
#pragma unroll
          for (int k = 0; k < 16; k++) {
            if (2 * k >= k0 && 2 * k < k1) tail += v[k].x;
            if (2 * k + 1 >= k0 && 2 * k + 1 < k1) tail += v[k].y;
          }
        }
      }
      double tau = 0, beta = c0, den = 0, nz = 0;
      if (tail != 0.0) {
        double b = sqrt(c0 * c0 + tail);
        if (c0 >= 0) b = -b;
        tau = (b - c0) / b;
        beta = b;
        den = c0 - b;
        nz = 1;
      }
      if (lane == 0) {
        sc[0] = tau;
        sc[1] = den;
        sc[2] = nz;
        AT(s + 1, s) = beta;
        Rf[(unsigned)(s * n + n - 1)] = tau;
      }
    }
    lds_barrier();
    const double den = sc[1];
    const int r = s + 2 + t;
    if (r < n) {
      const double e = sc[2] != 0.0 ? xc[r] / den : 0.0;
      tun[r].y = e;
      Rf[(unsigned)(s * n + t)] = e;
      AT(r, s) = 0.0;  // matrixH(): Hessenberg part only
    }
    return sc[0];
  };

  // the resident columns back to global memory, rows from r1 on
  auto flush = [&](int r1) {
    for (int r = r1 + wave; r < n; r += NW)
      for (int c = max(cK, r1) + lane; c < n; c += 64) AT(r, c) = RES(r, c);
  };
  // resident columns of R rows
  auto columns = [](int R) { return SMALL ? 32 : R <= 128 ? 128 : R <= 170 ? 96 : 64; };
  // residency for rows r1..n-1
  auto reside = [&](int r1) {
    K = columns(n - r1);
    cK = max(n - K, 0);
    r0 = r1;
    for (int ra = r1 + wave; ra < n; ra += 4 * NW) {
      double v[4][2];
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int j = 0; j < 2; j++) v[k][j] = AT(min(ra + NW * k, n - 1), min(cK + lane + 64 * j, n - 1));
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          if (ra + NW * k < n && cK + lane + 64 * j < n && lane + 64 * j < K) RES(ra + NW * k, cK + lane + 64 * j) = v[k][j];
    }
  };

  // Column pass after step i (i = -1: the left dot of step 0 alone, with
  // zero factors).
  auto colpass = [&](int i) {
    const int s = i + 1;                   // the step whose left dot this is
    const int ms = n - s - 2;              // its inner terms: rows s+2..n-1
    const int ns = max(cK - (i + 2), 0);   // streamed columns, whole waves ending at cK
    const int nsw = (ns + 31) / 32;
    const bool stream = wave < nsw;
    const int c = stream ? cK - 32 * (nsw - wave) + (lane >> 1) : max(cK, i + 2) + 32 * (wave - nsw) + (lane >> 1);
    const int h = lane & 1;
    const bool act = c >= i + 2 && c < n;
    if (__ballot(act) == 0) return;
    const int cs = min(max(c, i + 2), n - 1);  // in range; lanes without a column compute along
    const double2 own = twe[cs];
    const double wl = i >= 0 ? own.x : 0.0, f = i >= 0 ? own.y : 0.0;
    const bool packet = cs - (i + 2) < ((n - s - 1) & ~1);
    const bool np = __ballot(!packet) != 0;
    const long L = (long)(s + 2) * n + (s + 1);  // bottom^T(0,0) in row-major storage
    const int skip = ((L & 1) && odd_n && ms > 0) ? 1 : 0;
    const int bound = ms > 0 ? ((ms - skip) / 4) * 4 + skip : 0;
    double acc = 0.0, top = 0.0, x0 = 0.0;
    const int ro = s + 2;  // row of inner term 0
    auto run = [&](auto st) __attribute__((always_inline)) {
      constexpr bool S = decltype(st)::value;
      // one row: A = H A (streamed; the row pass has done it for resident
      // columns), A = A H; stored
      auto upd = [&](int r, double v, double tu) {
        if (S) v = v - lf[r] * wl;
        return v - tu * f;
      };
      auto get = [&](int r) { return S ? (double)AT(r, cs) : RES(r, cs); };
      auto put = [&](int r, double v) {
        if (!act) return;
        if (S) AT(r, cs) = v;
        else RES(r, cs) = v;
      };
      // both lanes of a pair compute the rows outside the groups; lane 0 stores
      if (i >= 0) {
        const double v = upd(i + 1, get(i + 1), tun[i + 1].x);  // this row leaves the active block
        if (act && h == 0) AT(i + 1, cs) = v;
      }
      top = get(s + 1);
      if (i >= 0) {
        top = upd(s + 1, top, tun[s + 1].x);
        if (h == 0) put(s + 1, top);
      }
      if (skip) {
        const double2 q = tun[ro];
        const double v = upd(ro, get(ro), q.x);
        if (h == 0) put(ro, v);
        x0 = v * q.y;
      }
      auto group = [&](const double *p) {  // the pair's four products in Eigen's order
        if (np) {  // a wave with the odd last column
          const double q0 = lane_xor1(p[0]), q1 = lane_xor1(p[1]);
          const double sh = p[0] + (odd_n ? q1 : p[1]);
          const double sp = acc + (sh + lane_xor1(sh));
          // lane 0's view: its own first pair, the other lane's second pair
          const double a = p[0], b = odd_n ? q1 : p[1], c2 = q0, d = odd_n ? p[1] : q1;
          const double sl = (((acc + a) + b) + c2) + d;
          acc = packet ? sp : sl;
        } else {
          const double sh = p[0] + (odd_n ? lane_xor1(p[1]) : p[1]);
          acc = acc + (sh + lane_xor1(sh));
        }
      };
      int g = skip;
      for (; g + 16 <= bound; g += 16) {
        double v[8], p[8];
        double2 q[8];
        const int rr = ro + g + 2 * h;
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = get(rr + (k >> 1) * 4 + (k & 1));
#pragma unroll
        for (int k = 0; k < 8; k++) q[k] = tun[rr + (k >> 1) * 4 + (k & 1)];
#pragma unroll
        for (int k = 0; k < 8; k++) {
          v[k] = upd(rr + (k >> 1) * 4 + (k & 1), v[k], q[k].x);
          p[k] = v[k] * q[k].y;
        }
#pragma unroll
        for (int k = 0; k < 8; k++) put(rr + (k >> 1) * 4 + (k & 1), v[k]);
#pragma unroll
        for (int k = 0; k < 8; k += 2) group(p + k);
      }
      for (; g < bound; g += 4) {
        double v[2], p[2];
        const int rr = ro + g + 2 * h;
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const double2 q = tun[rr + k];
          v[k] = upd(rr + k, get(rr + k), q.x);
          p[k] = v[k] * q.y;
        }
#pragma unroll
        for (int k = 0; k < 2; k++) put(rr + k, v[k]);
        group(p);
      }
      for (int j = bound; j < ms; j++) {
        const double2 q = tun[ro + j];
        const double v = upd(ro + j, get(ro + j), q.x);
        if (h == 0) put(ro + j, v);
        acc = acc + v * q.y;
      }
    };
    if (stream) run(std::true_type());
    else run(std::false_type());
    if (skip) acc = acc + x0;
    if (act && h == 0) twe[c] = double2{acc + top, tun[c].y};
  };

  // step 0's reflector and left dot
  for (int r = t; r < NMAX; r += 64 * NW) tun[r] = double2{0.0, 0.0};
  for (int r = t; r < n; r += 64 * NW) {
    const double x = AT(r, 0);
    xc[r] = x;
    if (r >= 1) tile[((r - 1) >> 5) * HTW + ((r - 1) & 31)] = x * x;
    lf[r] = 0.0;
  }
  reside(1);
  __syncthreads();
  double tau = reflector(0, 1);
  __syncthreads();
  colpass(-1);
  __syncthreads();
  for (int i = 0; i + 2 < n; ++i) {
    const int rem = n - i - 1, m = rem - 1, asz = m & ~1;
    if (columns(rem) != K) {  // fewer rows: more resident columns
      flush(i + 1);
      __syncthreads();
      reside(i + 1);
      __syncthreads();
    }
    // ---- row pass: row r, lane parity par (terms j of that parity; parity 1 also column i+1)
    if (i + 1 + 32 * wave < n) {
      const int rl = lane >> 1, par = lane & 1;
      const int r = i + 1 + 32 * wave + rl, rc = min(r, n - 1);
      const double fac = rc == i + 1 ? tau : tau * tun[rc].y;
      if (par == 0 && r < n) lf[r] = fac;
      double l = 0.0, col0 = 0.0;
      const int U = cK - (i + 1);  // streamed columns, column i+1 first
      if (U > 0) {
        double *tl = tile + wave * HTW;
        const int lr = lane >> 3, lc = lane & 7;
        // 32 rows x 32 columns from column i+1+u0: one lane offset per eight
        // rows; the columns past U are resident ones, so still in the matrix
        unsigned go[4];
#pragma unroll
        for (int k = 0; k < 4; k++) go[k] = (unsigned)(min(i + 1 + 32 * wave + 8 * k + lr, n - 1) * n + i + 1 + lc);
        auto load = [&](int u0, double *d) {
          gptr<const double> g = A + u0;
#pragma unroll
          for (int q = 0; q < 4; q++)
#pragma unroll
            for (int k = 0; k < 4; k++) d[4 * q + k] = (g + 8 * q)[go[k]];
        };
        double *tw = tl + lr * HT8 + lc;
        const double *tr = tl + rl * HT8 + 1 - par;
        const double2 *ob = twe + i + 2 - par;
        double v[16], nx[16];
        load(0, v);
        for (int u0 = 0; u0 < U; u0 += 32) {
          if (u0 + 32 < U) load(u0 + 32, nx);
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int ub = u0 + 8 * q;
            if (ub < U) {
              wave_sync();
#pragma unroll
              for (int k = 0; k < 4; k++) tw[8 * k * HT8] = v[4 * q + k];
              wave_sync();
              double a[4];
              double2 o[4];
#pragma unroll
              for (int x = 0; x < 4; x++) {
                a[x] = tr[2 * x];
                o[x] = ob[ub + 2 * x];
              }
              if (ub > 0 && ub + 8 <= U) {
#pragma unroll
                for (int x = 0; x < 4; x++) l = l + (a[x] - fac * o[x].x) * o[x].y;
              } else {  // column i+1, which is no term; columns past U
#pragma unroll
                for (int x = 0; x < 4; x++) {
                  const double w = a[x] - fac * o[x].x;
                  const double ln = l + w * o[x].y;
                  const int u = ub + 2 * x + 1 - par;
                  if (x == 0) col0 = (ub == 0 && par) ? w : col0;
                  l = (u < U && (x > 0 || ub > 0 || !par)) ? ln : l;
                }
              }
            }
          }
#pragma unroll
          for (int k = 0; k < 16; k++) v[k] = nx[k];
        }
      } else if (par) {
        col0 = RES(rc, i + 1) - fac * twe[i + 1].x;
      }
      // resident columns: terms j0.. of this parity
      const int j0 = max(U - 1, 0);
      int j = j0 + ((j0 ^ par) & 1);
      for (; j + 14 < asz; j += 16) {
        double a[8];
        double2 o[8];
#pragma unroll
        for (int x = 0; x < 8; x++) a[x] = RES(rc, i + 2 + j + 2 * x);
#pragma unroll
        for (int x = 0; x < 8; x++) o[x] = twe[i + 2 + j + 2 * x];
#pragma unroll
        for (int x = 0; x < 8; x++) {
          a[x] = a[x] - fac * o[x].x;
          l = l + a[x] * o[x].y;
        }
        if (r < n)
#pragma unroll
          for (int x = 0; x < 8; x++) RES(rc, i + 2 + j + 2 * x) = a[x];
      }
      {
        double a[8];
        double2 o[8];
#pragma unroll
        for (int x = 0; x < 8; x++) {
          const int c = min(i + 2 + j + 2 * x, n - 1);
          a[x] = RES(rc, c);
          o[x] = twe[c];
        }
#pragma unroll
        for (int x = 0; x < 8; x++) {
          a[x] = a[x] - fac * o[x].x;
          const double ln = l + a[x] * o[x].y;
          l = j + 2 * x < asz ? ln : l;
          if (r < n && j + 2 * x < asz) RES(rc, i + 2 + j + 2 * x) = a[x];
        }
      }
      double last = 0.0;
      if ((m & 1) && par == 0) {  // the odd last term, column n-1
        const double2 o = twe[n - 1];
        const double v = RES(rc, n - 1) - fac * o.x;
        if (r < n) RES(rc, n - 1) = v;
        last = v * o.y;
      }
      const double l1 = lane_xor1(l), cc0 = lane_xor1(col0);
      wave_sync();  // the tile's reads are done: it now holds the squares
      if (par == 0 && r < n) {
        double tmp = 0.0;
        if (asz > 0) tmp = tmp + (l + l1);
        if (m & 1) tmp = tmp + last;
        const double tt = (0.0 + tmp) + cc0;
        const double tuv = tau * tt;
        tun[r].x = tuv;
        const double x = cc0 - tuv;  // column i+1 of A = A H: (tau*tmp) * 1
        xc[r] = x;
        tile[wave * HTW + rl] = x * x;
        if (r == i + 1) AT(r, i + 1) = x;
      }
    }
    lds_barrier();
    const double tau_n = reflector(i + 1, i + 1);
    lds_barrier();
    colpass(i);
    if (cK > i + 2) __syncthreads();  // streamed columns were stored
    else lds_barrier();
    tau = tau_n;
  }
  flush(n - 1);
}
#undef RES
#undef AT

// The rows above the active block, after k_har_hess: row r (r <= n-3) receives
// the right reflectors of steps r..n-3 in order, with the operations of the
// reduction's own rows: the row dot in the RowMajor GEMV order, tu = tau * (dot
// + A(r, i+1)), A(r, i+1) -= tu, A(r, c) -= tu * ess[c-i-2].  Rows are
// independent, so a wave takes 32 of them on its own, two lanes per row (the
// even and the odd columns: the two lanes of the GEMV, which swap roles every
// step), staged in LDS with their live columns; the update of step i-1 and the
// dot of step i share one pass over the row.  As the last part of k_har_hess,
// with 68 rows at a time and two block barriers per step, this took a third
// of that kernel: 3.2M of 9.9M cycles for 238 tones.
constexpr int RWS = 32;  // rows per wave
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1)))
k_har_hess_rows(const HarDesc *hd, const int *order) {
  __shared__ double rows[RWS * 257];
  __shared__ double E[2][2][128];  // essential part of step s by column: [s & 1][c & 1][c >> 1]
  const int angle = blockIdx.x;
  const HarDesc H = hd[order[blockIdx.y]];
  const int n = __builtin_amdgcn_readfirstlane(*H.ng);
  const int r0 = RWS * blockIdx.z;
  if (r0 >= n - 2) return;
  gptr<double> A = to_global(H.Q + (long)angle * n * n);
  gptr<const double> Rf = to_global((const double *)H.P + (long)angle * n * n);
  const int lane = threadIdx.x, rr = lane >> 1, cp = lane & 1;
  const int nr = min(RWS, n - 2 - r0), cb = r0 + 1, wd = n - cb, wp = wd | 1;
  for (int ra = 0; ra < nr; ra += 4) {
    double v[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int k = 0; k < 4; k++) v[q][k] = A[(unsigned)((r0 + min(ra + q, nr - 1)) * n + cb + min(lane + 64 * k, wd - 1))];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (ra + q < nr && lane + 64 * k < wd) rows[(ra + q) * wp + lane + 64 * k] = v[q][k];
  }
  double *row = rows + rr * wp - cb;  // row[c]; rows past nr compute along in their own space
  auto fetch = [&](int i, double *e, double &tau) {
    const int m = n - i - 2;
#pragma unroll
    for (int k = 0; k < 4; k++) e[k] = Rf[(unsigned)(i * n + min(lane + 64 * k, max(m - 1, 0)))];
    tau = Rf[(unsigned)(i * n + n - 1)];
  };
  auto deposit = [&](int i, const double *e) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int c = i + 2 + lane + 64 * k;
      if (c < n) E[i & 1][c & 1][c >> 1] = e[k];
    }
  };
  double tau, tu = 0;
  {
    double e[4];
    fetch(r0, e, tau);
    deposit(r0, e);
  }
  wave_sync();
  // pass i: the update of step i-1 and the dot of step i (i = n-2: the update
  // alone).  SEL: some rows have not started yet and keep their values.
  auto pass = [&](int i, auto sel) __attribute__((always_inline)) {
    constexpr bool SEL = decltype(sel)::value;
    const bool begun = r0 + rr < i;
    const double *ep = E[(i - 1) & 1][cp], *ec = E[i & 1][cp];
    double en[4], tau_n = 0;
    if (i + 1 <= n - 3) fetch(i + 1, en, tau_n);
    auto upd = [&](double v, double e) {
      const double w = v - tu * e;
      return SEL ? (begun ? w : v) : w;
    };
    if (begun && cp == (i & 1)) row[i] = row[i] - tu;
    double col0 = 0;
    if (cp == ((i + 1) & 1)) {
      col0 = upd(row[i + 1], ep[(i + 1) >> 1]);
      row[i + 1] = col0;
    }
    if (i > n - 3) return;
    double l = 0;
    int c = i + 2 + ((i + 2 - cp) & 1);                    // this lane's first column
    const int nb = max(n - 2 - (i + 3) + 2, 0) / 2 / 8;    // full batches of eight columns of either parity
    struct Batch { double v[8], p[8], q[8]; };
    auto load = [&](int c, Batch &b) {
#pragma unroll
      for (int x = 0; x < 8; x++) b.v[x] = row[c + 2 * x];
#pragma unroll
      for (int x = 0; x < 8; x++) b.p[x] = ep[(c >> 1) + x];
#pragma unroll
      for (int x = 0; x < 8; x++) b.q[x] = ec[(c >> 1) + x];
    };
    auto work = [&](int c, Batch &b) {
#pragma unroll
      for (int x = 0; x < 8; x++) {
        b.v[x] = upd(b.v[x], b.p[x]);
        l = l + b.v[x] * b.q[x];
      }
#pragma unroll
      for (int x = 0; x < 8; x++) row[c + 2 * x] = b.v[x];
    };
    Batch a, b;
    if (nb > 0) load(c, a);
    for (int k = 0; k < nb; k += 2) {  // the next batch's reads in flight during this one's arithmetic
      if (k + 1 < nb) load(c + 16, b);
      work(c, a);
      c += 16;
      if (k + 1 < nb) {
        if (k + 2 < nb) load(c + 16, a);
        work(c, b);
        c += 16;
      }
    }
    // the rest up to column n-2 (at most eight per lane), then column n-1
#pragma unroll
    for (int x = 0; x < 8; x++) {
      const int cx = min(c + 2 * x, n - 1);
      a.v[x] = row[cx];
      a.p[x] = ep[cx >> 1];
      a.q[x] = ec[cx >> 1];
    }
    const bool own = cp == ((n - 1) & 1);
    double vl = row[n - 1];
    const double pl = ep[(n - 1) >> 1], ql = ec[(n - 1) >> 1];
#pragma unroll
    for (int x = 0; x < 8; x++) {
      const bool in = c + 2 * x <= n - 2;
      const double w = upd(a.v[x], a.p[x]);
      const double ln = l + w * a.q[x];
      l = in ? ln : l;
      if (in) row[c + 2 * x] = w;
    }
    double tl = 0;
    if (own) {
      vl = upd(vl, pl);
      row[n - 1] = vl;
      tl = vl * ql;
    }
    const bool odd_m = (n - i - 2) & 1;  // an odd last term stays apart
    if (own && !odd_m) l = l + tl;
    const double lx = lane_xor1(l), tx = lane_xor1(tl), cx = lane_xor1(col0);
    double tmp = 0.0 + (l + lx);
    if (odd_m) tmp = tmp + (own ? tl : tx);
    tu = tau * ((0.0 + tmp) + (cp == ((i + 1) & 1) ? col0 : cx));
    if (i + 1 <= n - 3) deposit(i + 1, en);
    tau = tau_n;
    wave_sync();
  };
  int i = r0;
  for (; i <= n - 2 && i < r0 + RWS; i++) pass(i, std::true_type());
  for (; i <= n - 2; i++) pass(i, std::false_type());
  wave_sync();
  for (int ra = 0; ra < nr; ra++)
    for (int c = lane; c < wd; c += 64) A[(unsigned)((r0 + ra) * n + cb + c)] = rows[ra * wp + c];
}

// Francis QR on the Hessenberg matrix left in H.Q by k_har_hess, for launches
// of many matrices: one wave per (angle, image), sixteen per CU.  The Schur
// iteration is a chain of dependent steps, so many chains with a small LDS
// window each keep the CU busy; k_har_schur below serves smaller launches.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
k_har_qr(const HarDesc *hd, const int *order, const int *pick) {
  if (pick && *pick != 0) return;  // uniform: k_har_schur takes the launch
  constexpr int RS = 2;   // window rows per pass of the wave (32 columns per row)
  constexpr int CH = QW;  // rows above the window staged per chunk
  __shared__ double Rw[CH * QWP];
  __shared__ double rf[QB][4];
  __shared__ double sc[8];
  __shared__ int si[8];
  __shared__ int ired[8];
  __shared__ double dred[8];
  __shared__ int s_iu;
  const int angle = blockIdx.x;
  const HarDesc H = hd[order[blockIdx.y]];
  const int n = *H.ng;
  gptr<double> A = to_global(H.Q + (long)angle * n * n);
  const int t = threadIdx.x;
#define AT(r, c) A[(long)(r) * n + (c)]
  // ---- real Schur form (RealSchur::compute without U); left updates are
  // restricted to columns <= iu (entries right of the active window are
  // never read again), right updates cover rows 0..min(iu,k+3) as in Eigen.
  // RealSchur::computeNormOfT (RealSchur.h:274-285) on row-major storage:
  // each row segment T(j, max(j-1,0)..n-1) is a contiguous Eigen redux, and
  // the segment sums are added row by row
  double *segs = Rw;  // the window buffer is free until the first window
  for (int j = t; j < n; j += blockDim.x) {
    const int k0 = j - 1 > 0 ? j - 1 : 0;
    gptr<const double> row = A + ((long)j * n + k0);
    segs[j] = eigen_redux(n - k0, (int)(((long)j * n + k0) & 1), [&](int k) { return fabs(row[k]); });
  }
  __syncthreads();
  if (t == 0) {
    double sn = 0;
    for (int j = 0; j < n; j++) sn += segs[j];
    dred[0] = sn;
  }
  __syncthreads();
  const double norm = dred[0];
  const double eps = kDblEps;
  // decision state (iu, iteration counts, exceptional shift) lives in
  // thread 0; the block follows through s_iu / si / sc
  int iu = n - 1, iter = 0, totalIter = 0;
  double exshift = 0;
  double work = 0;  // thread 0: flops of the updates issued (12 per 3-vector, 6 per 2-vector / rotation)
  if (t == 0) s_iu = n - 1;
  __syncthreads();
  while (norm != 0) {
    __syncthreads();  // every thread has consumed the previous decision
    const int iub = s_iu;
    if (iub < 0) break;
    // findSmallSubdiagEntry: the largest res in (0, iu] whose subdiagonal
    // entry is negligible, else 0 -- every candidate tested at once
    // (a lane's candidates are res = iub - t - 64k, k < 4 since n <= 256: all
    // their entries are loaded at once, then tested in descending order)
    int cand = 0;
    {
      double dd0[4] = {0, 0, 0, 0}, dd1[4] = {0, 0, 0, 0}, sd[4] = {0, 0, 0, 0};
      if (n >= 2)  // otherwise there is no candidate
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int res = min(max(iub - t - 64 * k, 1), n - 1);  // in range; unused when res <= 0
          dd0[k] = AT(res - 1, res - 1);
          dd1[k] = AT(res, res);
          sd[k] = AT(res, res - 1);
        }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int res = iub - t - 64 * k;
        if (res > 0 && cand == 0) {
          double s = fabs(dd0[k]) + fabs(dd1[k]);
          if (s == 0.0) s = norm;
          if (fabs(sd[k]) < eps * s) cand = res;
        }
      }
    }
    const int il = block_reduce(cand, MaxOp(), ired);
    if (t == 0) {
      int action = 3;
      if (il == iu) {  // one root
        AT(iu, iu) = AT(iu, iu) + exshift;
        if (iu > 0) AT(iu, iu - 1) = 0;
        iu--; iter = 0;
        action = 0;
      } else if (il == iu - 1) {  // two roots (RealSchur::splitOffTwoRows)
        action = 1;
        const double p = 0.5 * (AT(iu - 1, iu - 1) - AT(iu, iu));
        const double q = p * p + AT(iu, iu - 1) * AT(iu - 1, iu);
        AT(iu, iu) += exshift;
        AT(iu - 1, iu - 1) += exshift;
        si[3] = q >= 0;
        if (q >= 0) {
          const double z = sqrt(fabs(q));
          const double pp = (p >= 0) ? p + z : p - z, qq = AT(iu, iu - 1);
          double c, s;  // JacobiRotation::makeGivens, real case
          if (qq == 0) { c = pp < 0 ? -1 : 1; s = 0; }
          else if (pp == 0) { c = 0; s = qq < 0 ? 1 : -1; }
          else if (fabs(pp) > fabs(qq)) {
            const double tt = qq / pp;
            double u = sqrt(1 + tt * tt);
            if (pp < 0) u = -u;
            c = 1 / u; s = -tt * c;
          } else {
            const double tt = pp / qq;
            double u = sqrt(1 + tt * tt);
            if (qq < 0) u = -u;
            s = -1 / u; c = -tt * s;
          }
          sc[1] = c; sc[2] = s;
          for (int j = iu - 1; j <= iu; j++) {  // rot.adjoint() on the left, columns <= iu
            const double xv = AT(iu - 1, j), yv = AT(iu, j);
            AT(iu - 1, j) = c * xv - s * yv;
            AT(iu, j) = s * xv + c * yv;
          }
        }
        si[1] = iu;  // rows 0..iu get the right rotation
        if (q >= 0) work += 6.0 * (2 + iu + 1);
        iu -= 2; iter = 0;
      } else {  // Francis QR step (RealSchur::computeShift)
        double sh0 = AT(iu, iu), sh1 = AT(iu - 1, iu - 1), sh2 = AT(iu, iu - 1) * AT(iu - 1, iu);
        double shift_amt = 0;
        int shift_kind = 0;
        if (iter == 10) {
          exshift += sh0;
          shift_kind = 1; shift_amt = sh0;
          const double s = fabs(AT(iu, iu - 1)) + fabs(AT(iu - 1, iu - 2));
          sh0 = 0.75 * s; sh1 = 0.75 * s; sh2 = -0.4375 * s * s;
        }
        if (iter == 30) {
          double s = (sh1 - sh0) / 2.0;
          s = s * s + sh2;
          if (s > 0) {
            s = sqrt(s);
            if (sh1 < sh0) s = -s;
            s = s + (sh1 - sh0) / 2.0;
            s = sh0 - sh2 / s;
            exshift += s;
            shift_kind = 2; shift_amt = s;
            sh0 = sh1 = sh2 = 0.964;
          }
        }
        iter++; totalIter++;
        if (totalIter > 40 * n) action = 3;
        else {
          action = 2;
          if (shift_kind) work += iu + 1;
          si[4] = shift_kind;
          sc[3] = shift_amt;
          sc[4] = sh0; sc[5] = sh1; sc[6] = sh2;
          si[5] = iu;
        }
      }
      si[0] = action;
      s_iu = action == 3 ? -1 : iu;
    }
    __syncthreads();
    const int action = si[0];
    if (action == 3) break;
    if (action == 0) continue;
    if (action == 1) {
      const int iu2 = si[1];
      if (si[3]) {
        const double c = sc[1], s = sc[2];
        for (int r = t; r <= iu2; r += blockDim.x) {  // rot on the right, rows 0..iu
          const double xv = AT(r, iu2 - 1), yv = AT(r, iu2);
          AT(r, iu2 - 1) = c * xv - s * yv;
          AT(r, iu2) = s * xv + c * yv;
        }
        __syncthreads();
        if (t == 0) AT(iu2, iu2 - 1) = 0;
      }
      if (t == 0 && iu2 > 1) AT(iu2 - 1, iu2 - 2) = 0;
      continue;  // the loop head synchronises
    }
    // ---- Francis QR step on the window [il, iuq]
    const int iuq = si[5];
    if (si[4]) {
      const double amt = sc[3];
      for (int i = t; i <= iuq; i += blockDim.x) AT(i, i) -= amt;
      __syncthreads();
    }
    // initFrancisQRStep: the largest im in (il, iuq-2] passing the
    // small-subdiagonal test, else il -- every candidate tested at once
    const double sh0 = sc[4], sh1 = sc[5], sh2 = sc[6];
    // (candidates m = iuq - 2 - t - 64k, k < 4: entries loaded at once, then
    // tested in descending order)
    cand = il;
    {
      double tmm[4] = {0, 0, 0, 0}, t10[4] = {0, 0, 0, 0}, t01[4] = {0, 0, 0, 0}, t11[4] = {0, 0, 0, 0};
      double t21[4] = {0, 0, 0, 0}, tm1[4] = {0, 0, 0, 0}, tpp[4] = {0, 0, 0, 0};
      if (n >= 4)  // otherwise there is no candidate m > il >= 0 with m + 2 <= iuq
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int m = min(max(iuq - 2 - t - 64 * k, 1), n - 3);  // in range; unused when m <= il
        tmm[k] = AT(m, m);
        t10[k] = AT(m + 1, m);
        t01[k] = AT(m, m + 1);
        t11[k] = AT(m + 1, m + 1);
        t21[k] = AT(m + 2, m + 1);
        tm1[k] = AT(m, m - 1);
        tpp[k] = AT(m - 1, m - 1);
      }
      bool found = false;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int m = iuq - 2 - t - 64 * k;
        if (m > il && !found) {
          const double Tmm = tmm[k];
          const double r = sh0 - Tmm, s = sh1 - Tmm;
          const double v0 = (r * s - sh2) / t10[k] + t01[k];
          const double v1 = t11[k] - Tmm - r - s;
          const double v2 = t21[k];
          const double lhs = tm1[k] * (fabs(v1) + fabs(v2));
          const double rhs = v0 * (fabs(tpp[k]) + fabs(Tmm) + fabs(t11[k]));
          if (fabs(lhs) < eps * rhs) { cand = m; found = true; }
        }
      }
    }
    const int im = block_reduce(cand, MaxOp(), ired);
    if (t == 0)
      for (int k = im; k <= iuq - 2; k++) work += 12.0 * ((iuq - k + 1) + ((iuq < k + 3 ? iuq : k + 3) + 1));
    double fv0, fv1, fv2;
    {
      const double Tmm = AT(im, im);
      const double r = sh0 - Tmm, s = sh1 - Tmm;
      fv0 = (r * s - sh2) / AT(im + 1, im) + AT(im, im + 1);
      fv1 = AT(im + 1, im + 1) - Tmm - r - s;
      fv2 = AT(im + 2, im + 1);
    }
    // Bulge chase in windows of QB steps.  Window steps [k0, k1) read and
    // update only entries inside R = [a, b) x [a, b) (a = k0-1, b = k1+3),
    // which live in LDS while wavefront 0 chases the bulge through them;
    // afterwards the window's reflectors are applied, in step order, to the
    // strips outside R (rows k0..k1+1 right of R: left reflectors only;
    // columns k0..k1+1 above R: right reflectors only).  Every entry
    // therefore receives the same reflectors in the same order as in the
    // unwindowed chase.
    for (int k0 = im; k0 <= iuq - 2; k0 += QB) {
      const int k1 = (k0 + QB < iuq - 1) ? k0 + QB : iuq - 1;
      const int a = k0 - 1 > 0 ? k0 - 1 : 0;
      const int b = (k1 + 3 < iuq + 1) ? k1 + 3 : iuq + 1;
      const int wd = b - a;
      {  // 32 x 32 tile, RS rows per block pass, all loads in flight
        int rb = t >> 5;
        asm volatile("" : "+v"(rb));  // per-row values are formed here, not hoisted out of the sweep loop
        const int cl = t & 31;
        const int cc = min(cl, wd - 1);  // out-of-window lanes re-read in-window entries (unused)
        double v[QW / RS];
#pragma unroll
        for (int it = 0; it < QW / RS; it++) v[it] = A[(unsigned)((a + min(rb + RS * it, wd - 1)) * n + a + cc)];
#pragma unroll
        for (int it = 0; it < QW / RS; it++) {
          const int r = rb + RS * it;
          if (r < wd && cl < wd) Rw[r * QWP + cl] = v[it];
        }
      }
      __syncthreads();
#define RW(r, c) Rw[((r) - a) * QWP + ((c) - a)]
      if (t < 64) {
        for (int k = k0; k < k1; ++k) {
          const bool first = (k == im);
          double x0, x1, x2;
          if (first) { x0 = fv0; x1 = fv1; x2 = fv2; }
          else { x0 = RW(k, k - 1); x1 = RW(k + 1, k - 1); x2 = RW(k + 2, k - 1); }
          // makeHouseholder of (x0, x1, x2), every lane
          double tail = 0;
          tail += x1 * x1;
          tail += x2 * x2;
          double tau = 0, e0 = 0, e1 = 0, beta = x0;
          if (tail != 0.0) {
            double bb = sqrt(x0 * x0 + tail);
            if (x0 >= 0) bb = -bb;
            e0 = x1 / (x0 - bb);
            e1 = x2 / (x0 - bb);
            tau = (bb - x0) / bb;
            beta = bb;
          }
          wave_sync();
          if (t == 0) {
            rf[k - k0][0] = beta != 0 ? tau : 0.0;
            rf[k - k0][1] = e0;
            rf[k - k0][2] = e1;
            rf[k - k0][3] = beta != 0 ? 1.0 : 0.0;
          }
          if (beta != 0) {
            if (t == 0) {
              if (first && k > il) RW(k, k - 1) = -RW(k, k - 1);
              else if (!first) RW(k, k - 1) = beta;
            }
            const int c = k + t;
            if (c < b) {
              double tt = e0 * RW(k + 1, c);
              tt += e1 * RW(k + 2, c);
              tt += RW(k, c);
              RW(k, c) -= tau * tt;
              RW(k + 1, c) -= (tau * e0) * tt;
              RW(k + 2, c) -= (tau * e1) * tt;
            }
            wave_sync();
            const int rlast = (iuq < k + 3 ? iuq : k + 3);
            const int r = a + t;
            if (r <= rlast) {
              double tt = RW(r, k + 1) * e0;
              tt += RW(r, k + 2) * e1;
              tt += RW(r, k);
              RW(r, k) -= tau * tt;
              RW(r, k + 1) -= (tau * tt) * e0;
              RW(r, k + 2) -= (tau * tt) * e1;
            }
            wave_sync();
          }
        }
      }
      __syncthreads();
      // the window's steps whose reflector is applied (beta != 0), one bit per
      // step: a uniform mask, so the strip loops branch on it without an LDS
      // round trip per step
      const unsigned long long fon = __ballot((t & 63) < QB && rf[min(t & 63, QB - 1)][3] != 0.0);
      for (int r = t >> 5; r < wd; r += RS)
        if ((t & 31) < wd) AT(a + r, a + (t & 31)) = Rw[r * QWP + (t & 31)];
#undef RW
      // strip right of R: rows k0 .. k1+1, columns b .. iuq (left reflectors).
      // Reflector q touches rows q..q+2 of the strip, so after it row q is
      // final: each thread streams down its column with a 3-value window.
      const int nstep = k1 - k0;
      for (int c = b + t; c <= iuq; c += blockDim.x) {
        gptr<double> p = A + ((long)k0 * n + c);
        double w[QB + 2];
        {
          gptr<const double> pl = p;  // running pointer: one live address
#pragma unroll
          for (int q = 0; q < QB + 2; q++) {
            w[q] = (q < nstep + 2) ? *pl : 0.0;
            pl += n;
          }
        }
        // every load has arrived before the first store: the stores below then
        // never stand in the way of a load's wait (the vector-memory counter
        // counts both)
        __builtin_amdgcn_s_waitcnt(0);
        gptr<double> ps = p;
        double u0 = w[0], u1 = w[1];
#pragma unroll
        for (int q = 0; q < QB; q++) {
          if (q < nstep) {
            double u2 = w[q + 2];
            if ((fon >> q) & 1) {
              const double tau = rf[q][0], e0 = rf[q][1], e1 = rf[q][2];
              double tt = e0 * u1;
              tt += e1 * u2;
              tt += u0;
              u0 -= tau * tt;
              u1 -= (tau * e0) * tt;
              u2 -= (tau * e1) * tt;
            }
            *ps = u0;
            ps += n;
            u0 = u1;
            u1 = u2;
          }
          __asm__ volatile("" ::: "memory");  // keep the reflector loads step by step
        }
        ps[0] = u0;
        ps[n] = u1;
      }
      // strip above R: rows 0 .. a-1, columns k0 .. k1+1 (right reflectors).
      // Staged through the (now free) window buffer in chunks of CH rows with
      // coalesced loads and stores; one lane streams each row through the
      // reflectors in LDS.
      __syncthreads();
      for (int r0 = 0; r0 < a; r0 += CH) {  // a chunk fills at most the window buffer
        const int nr = (a - r0 < CH) ? a - r0 : CH;
        const int nc = nstep + 2;
        {
          int rb = t >> 5;
          asm volatile("" : "+v"(rb));
          const int cl = t & 31;
          const int cc = min(cl, nc - 1);
          double v[CH / RS];
#pragma unroll
          for (int it = 0; it < CH / RS; it++) v[it] = A[(unsigned)((r0 + min(rb + RS * it, nr - 1)) * n + k0 + cc)];
#pragma unroll
          for (int it = 0; it < CH / RS; it++) {
            const int rr = rb + RS * it;
            if (rr < nr && cl < nc) Rw[rr * QWP + cl] = v[it];
          }
        }
        __syncthreads();
        if (t < nr) {
          // the row's entries first (LDS reads in flight together; entries
          // past the window's columns are read but left as they are)
          double *row = Rw + t * QWP;
          double x[QB + 2];
#pragma unroll
          for (int q = 0; q < QB + 2; q++) x[q] = row[q];
          double u0 = x[0], u1 = x[1];
#pragma unroll
          for (int q = 0; q < QB; q++) {
            if (q < nstep) {
              double u2 = x[q + 2];
              if ((fon >> q) & 1) {
                const double tau = rf[q][0], e0 = rf[q][1], e1 = rf[q][2];
                double tt = u1 * e0;
                tt += u2 * e1;
                tt += u0;
                u0 -= tau * tt;
                u1 -= (tau * tt) * e0;
                u2 -= (tau * tt) * e1;
              }
              row[q] = u0;
              u0 = u1;
              u1 = u2;
            }
            __asm__ volatile("" ::: "memory");  // the reflector reads step by step
          }
          row[nstep] = u0;
          row[nstep + 1] = u1;
        }
        __syncthreads();
        for (int rr = t >> 5; rr < nr; rr += RS)
          if ((t & 31) < nc) AT(r0 + rr, k0 + (t & 31)) = Rw[rr * QWP + (t & 31)];
        __syncthreads();
      }
    }
    if (t == 0) {
      double x[2] = {AT(iuq - 1, iuq - 2), AT(iuq, iuq - 2)};
      double e1[1], tau, beta;
      make_hh(x, 2, e1, &tau, &beta);
      si[6] = beta != 0;
      if (beta != 0) { AT(iuq - 1, iuq - 2) = beta; work += 6.0 * (2 + iuq + 1); }
      sc[3] = tau; sc[7] = e1[0];
    }
    __syncthreads();
    if (si[6]) {
      const double tau = sc[3], e0 = sc[7];
      if (t == 0)
        for (int c = iuq - 1; c <= iuq; c++) {
          double tt = e0 * AT(iuq, c);
          tt += AT(iuq - 1, c);
          AT(iuq - 1, c) -= tau * tt;
          AT(iuq, c) -= (tau * e0) * tt;
        }
      __syncthreads();
      for (int r = t; r <= iuq; r += blockDim.x) {
        double tt = AT(r, iuq) * e0;
        tt += AT(r, iuq - 1);
        AT(r, iuq - 1) -= tau * tt;
        AT(r, iuq) -= (tau * tt) * e0;
      }
    }
    for (int i = im + 2 + t; i <= iuq; i += blockDim.x) {
      AT(i, i - 2) = 0;
      if (i > im + 2) AT(i, i - 3) = 0;
    }
  }
  __syncthreads();
  // eigenvalue 2 in Schur-diagonal order (EigenSolver::compute, EigenSolver.h:364-381)
  if (t == 0) {
    double f = 0.0;
    if (n >= 3) {
      int i = 0;
      double re2 = 0, im2 = 0;
      while (i < n && i <= 2) {
        if (i == n - 1 || AT(i + 1, i) == 0) {
          if (i == 2) { re2 = AT(i, i); im2 = 0; }
          ++i;
        } else {
          const double p = 0.5 * (AT(i, i) - AT(i + 1, i + 1));
          const double z = sqrt(fabs(p * p + AT(i + 1, i) * AT(i, i + 1)));
          if (i == 2) { re2 = AT(i + 1, i + 1) + p; im2 = z; }
          if (i + 1 == 2) { re2 = AT(i + 1, i + 1) + p; im2 = -z; }
          i += 2;
        }
      }
      f = (im2 == 0) ? sqrt(re2) : 0.0;
    }
    H.feat[angle * 14 + 13] = f;
    H.work[angle] = work;
  }
#undef AT
}

// ------------------------------------------------------- pipelined Schur form
// The same Francis iteration as k_har_qr with a matrix's chain of dependent
// steps on wave 0 alone, in registers, and everything off that chain on the
// other three waves of the block, one window of PB steps behind.
//
//   wave 0 (chase)   lane l holds the open rows k, k+1, k+2 of column k0 + l.
//     Per step: the reflector (the same in every lane), the left update of
//     all 64 columns at once, then the right update of rows k+1..k+3 on the
//     corner columns k..k+2, whose values are read from their lanes, updated
//     in every lane and put back.  Row k goes to LDS.  A step's only LDS read
//     is the row k+4, a step ahead; global memory is never touched.
//   waves 1-3        left updates of the columns right of the band, one column
//     per lane, following wave 0's reflectors through LDS (each carries its
//     step's number) with the rows of the window loaded ahead; right updates
//     of the previous window: its own PB rows and the rows above, through a
//     wave-private LDS transpose; the next window's rows into LDS.
//
// One block barrier per window.  Every entry receives the same reflectors in
// the same order, with the same operations, as in k_har_qr.  Subdiagonal
// entries live in LDS (sub[i] = T(i,i-1)); the bulge below them is never
// stored, as the iteration clears it at the end of every sweep.
//
// What bounds it: the chain, about 100 instructions of wave 0 per step, issued
// one per four cycles (an FP64 instruction's rate; dependent ones gain nothing
// on independent ones): about 650 cycles per step, 28,000 steps for 240 tones.  With
// one block of 256 threads chasing through an LDS window, as this kernel's
// predecessor did, a step took 2,500 cycles: three LDS round trips, three IEEE
// divisions and a square root with their scaling, and the strips in between.
constexpr int PB = 16;        // steps per window
constexpr int PWP = 65;       // padded row of a window buffer (64 columns)
constexpr int PT = 64;        // rows of a transpose buffer
constexpr int PTP = PB + 3;   // its padded row (odd)

__device__ __forceinline__ double lane_value(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | lo);
}

struct __align__(16) SchurRf {
  double tau, e0, e1;
  int gen, app;  // step number; whether the reflector is applied (beta != 0)
};

// steps 0, 1, .. while step(q) accepts, in groups of four up to lim (a
// multiple of four); returns how many were done
template <class Step, int... Q>
__device__ __forceinline__ int schur_steps(Step &step, int lim, std::integer_sequence<int, Q...>) {
  int done = 0;
  (void)(((Q % 4 != 0 || Q < lim) && step(std::integral_constant<int, Q>()) && (done = Q + 1, true)) && ...);
  return done;
}
typedef double schur_d2 __attribute__((ext_vector_type(2)));

// Right reflectors of a window applied to one row, row[0..PB+1] = columns
// k0..k1+1 (and on, unchanged): the steps whose bit is set in `on`, or all.
template <bool ALL>
__device__ __forceinline__ void schur_right(unsigned on, const SchurRf *rf, double *row) {
  double x[PB + 2];
#pragma unroll
  for (int q = 0; q < PB + 2; q++) x[q] = row[q];
  double u0 = x[0], u1 = x[1];
  double tau = rf[0].tau, e0 = rf[0].e0, e1 = rf[0].e1;
#pragma unroll
  for (int q = 0; q < PB; q++) {
    double ntau = 0, ne0 = 0, ne1 = 0;
    if (q + 1 < PB) {  // the next step's reflector during this step
      ntau = rf[q + 1].tau; ne0 = rf[q + 1].e0; ne1 = rf[q + 1].e1;
    }
    double u2 = x[q + 2];
    double tt = u1 * e0;
    tt += u2 * e1;
    tt += u0;
    const double w = tau * tt;
    double n0 = u0 - w, n1 = u1 - w * e0, n2 = u2 - w * e1;
    if (!ALL) {
      __asm__ volatile("" : "+v"(n0), "+v"(n1), "+v"(n2));  // selects, no branches
      const bool take = (int)(on << (31 - q)) < 0;
      n0 = take ? n0 : u0;
      n1 = take ? n1 : u1;
      n2 = take ? n2 : u2;
    }
    row[q] = n0;
    u0 = n1;
    u1 = n2;
    tau = ntau; e0 = ne0; e1 = ne1;
    __asm__ volatile("" ::: "memory");
  }
  row[PB] = u0;
  row[PB + 1] = u1;
}

// POLLS: how often a wave looks for another's result before it gives up
constexpr int SCHUR_POLLS = 1 << 24;  // most of a second
template <int NW, int POLLS = SCHUR_POLLS>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
k_har_schur(const HarDesc *hd, const int *order, const int *pick) {
  if (pick && *pick == 0) return;  // uniform: k_har_qr takes the launch
  // window t's buffer (t mod 3): slot j first holds row k0+3+j, which wave 0
  // reads at step j, then the finished row k0+j, which it writes at step j;
  // column k0 + l at l
  __shared__ double win[3][PB * PWP];
  __shared__ double tbuf[NW][PT * PTP];
  __shared__ SchurRf rf[2][PB];
  __shared__ double hand[2][3][64];  // open rows k1, k1+1, k1+2 of the next window's columns k1..k1+63
  __shared__ double dia[256], sup[256], sub[260];
  __shared__ double fin[3];          // last reflector of the sweep: tau, e0, applied
  __shared__ double dred;
  __shared__ unsigned long long wm[NW];
  const int angle = blockIdx.x;
  const HarDesc H = hd[order[blockIdx.y]];
  const int n = __builtin_amdgcn_readfirstlane(*H.ng);
  gptr<double> A = to_global(H.Q + (long)angle * n * n);
  // Which wave chases: two blocks share a CU (NW = 4), and their chases should
  // not share a SIMD.  A block's waves go to the SIMDs in the order 0, 2, 1, 3
  // from any start, so the first wave's SIMD and whether the block's LDS is the
  // CU's first tell which wave sits where; any answer is correct.
  __shared__ int s_rot;
  if (NW == 4 && threadIdx.x == 0) {
    const unsigned simd = (__builtin_amdgcn_s_getreg(4 | (31 << 11)) >> 4) & 3;   // HW_ID
    const unsigned base = __builtin_amdgcn_s_getreg(6 | (31 << 11)) & 0xfff;      // LDS_ALLOC
    const int pos = simd == 0 ? 0 : simd == 2 ? 1 : simd == 1 ? 2 : 3;
    s_rot = (pos + (base ? 2 : 0)) & 3;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = NW == 4 ? (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + __builtin_amdgcn_readfirstlane(s_rot)) & 3
                           : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = wave * 64 + lane;
#define AT(r, c) A[(unsigned)((r) * n + (c))]
  // RealSchur::computeNormOfT as in k_har_qr
  double *segs = win[0];
  if (t < n) {
    const int k0 = t - 1 > 0 ? t - 1 : 0;
    gptr<const double> row = A + ((long)t * n + k0);
    segs[t] = eigen_redux(n - k0, (int)(((long)t * n + k0) & 1), [&](int k) { return fabs(row[k]); });
    sub[t] = t > 0 ? AT(t, t - 1) : 0.0;
  }
  __syncthreads();
  if (t == 0) {
    double sn = 0;
    for (int j = 0; j < n; j++) sn += segs[j];
    dred = sn;
  }
  if (t < 2 * PB) rf[t / PB][t % PB].gen = 0;
  __syncthreads();
  const double norm = dred;
  const double eps = kDblEps;
  // a bound on the Frobenius norm, hence on every entry: reflections keep it,
  // and an exceptional shift s, |s| <= 2 |T|, adds at most 2 sqrt(n) of it
  double cap = norm;
  if (wave == 0) __builtin_amdgcn_s_setprio(3);  // the chain first where it shares its SIMD
  // decision state: every thread keeps it, from the same LDS values
  int iu = n - 1, iter = 0, totalIter = 0;
  double exshift = 0;
  double work = 0;
  int base = 0;  // steps published so far
  // highest thread index with a hit over the block (none: -1)
  auto highest = [&](bool hit) {
    const unsigned long long m = __ballot(hit);
    if (lane == 0) wm[wave] = m;
    __syncthreads();
    int r = -1;
#pragma unroll
    for (int w = 0; w < NW; w++)
      if (wm[w]) r = 64 * w + 63 - __clzll((long long)wm[w]);
    return __builtin_amdgcn_readfirstlane(r);
  };
  bool reload = true;
  while (norm != 0 && iu >= 0) {
    __syncthreads();  // the previous step's stores and LDS reads are complete
    iu = __builtin_amdgcn_readfirstlane(iu);  // the same in every thread: scalar branches and indices
    if (reload) {
      if (t <= iu) {
        dia[t] = AT(t, t);
        sup[t] = t < iu ? AT(t, t + 1) : 0.0;
      }
      reload = false;
      __syncthreads();
    }
    // findSmallSubdiagEntry: the largest res in (0, iu] with a negligible subdiagonal entry
    bool hit = false;
    if (t > 0 && t <= iu) {
      double s = fabs(dia[t - 1]) + fabs(dia[t]);
      if (s == 0.0) s = norm;
      hit = fabs(sub[t]) < eps * s;
    }
    const int il = max(highest(hit), 0);
    if (il == iu) {  // one root
      __syncthreads();
      if (t == 0) {
        const double d = dia[iu] + exshift;
        dia[iu] = d;
        AT(iu, iu) = d;
        if (iu > 0) sub[iu] = 0;
      }
      iu--;
      iter = 0;
      continue;
    }
    if (il == iu - 1) {  // two roots (RealSchur::splitOffTwoRows)
      const double p = 0.5 * (dia[iu - 1] - dia[iu]);
      const double q = p * p + sub[iu] * sup[iu - 1];
      const double a00 = dia[iu - 1] + exshift, a01 = sup[iu - 1], a10 = sub[iu], a11 = dia[iu] + exshift;
      __syncthreads();
      if (q >= 0) {
        const double z = sqrt(fabs(q));
        const double pp = (p >= 0) ? p + z : p - z, qq = a10;
        double c, s;  // JacobiRotation::makeGivens, real case
        if (qq == 0) { c = pp < 0 ? -1 : 1; s = 0; }
        else if (pp == 0) { c = 0; s = qq < 0 ? 1 : -1; }
        else if (fabs(pp) > fabs(qq)) {
          const double tt = qq / pp;
          double u = sqrt(1 + tt * tt);
          if (pp < 0) u = -u;
          c = 1 / u; s = -tt * c;
        } else {
          const double tt = pp / qq;
          double u = sqrt(1 + tt * tt);
          if (qq < 0) u = -u;
          s = -1 / u; c = -tt * s;
        }
        // left on columns iu-1, iu, then right on rows 0..iu
        const double b00 = c * a00 - s * a10, b10 = s * a00 + c * a10;
        const double b01 = c * a01 - s * a11, b11 = s * a01 + c * a11;
        if (t <= iu) {
          double xv, yv;
          if (t == iu - 1) { xv = b00; yv = b01; }
          else if (t == iu) { xv = b10; yv = b11; }
          else { xv = AT(t, iu - 1); yv = AT(t, iu); }
          const double l = c * xv - s * yv, rr = s * xv + c * yv;
          if (t < iu) AT(t, iu - 1) = l;
          AT(t, iu) = rr;
        }
        if (t == 0) { sub[iu] = 0; work += 6.0 * (2 + iu + 1); }
      } else if (t == 0) {
        AT(iu, iu) = a11;
        AT(iu - 1, iu - 1) = a00;
      }
      if (t == 0 && iu > 1) sub[iu - 1] = 0;
      iu -= 2;
      iter = 0;
      reload = true;
      continue;
    }
    // ---- Francis QR step (RealSchur::computeShift)
    double sh0 = dia[iu], sh1 = dia[iu - 1], sh2 = sub[iu] * sup[iu - 1];
    double amt = 0;
    int shift_kind = 0;
    if (iter == 10) {
      exshift += sh0;
      shift_kind = 1;
      amt = sh0;
      const double s = fabs(sub[iu]) + fabs(sub[iu - 1]);
      sh0 = 0.75 * s; sh1 = 0.75 * s; sh2 = -0.4375 * s * s;
    }
    if (iter == 30) {
      double s = (sh1 - sh0) / 2.0;
      s = s * s + sh2;
      if (s > 0) {
        s = sqrt(s);
        if (sh1 < sh0) s = -s;
        s = s + (sh1 - sh0) / 2.0;
        s = sh0 - sh2 / s;
        exshift += s;
        shift_kind = 2;
        amt = s;
        sh0 = sh1 = sh2 = 0.964;
      }
    }
    iter++;
    totalIter++;
    if (totalIter > 40 * n) break;
    __syncthreads();
    if (shift_kind) {
      cap *= 64;
      if (t <= iu) {
        const double d = dia[t] - amt;
        dia[t] = d;
        AT(t, t) = d;
      }
      work += iu + 1;
      __syncthreads();
    }
    // initFrancisQRStep: the largest im in (il, iu-2] passing the small-subdiagonal test, else il
    hit = false;
    if (t > il && t <= iu - 2) {
      const double Tmm = dia[t];
      const double r = sh0 - Tmm, s = sh1 - Tmm;
      const double v0 = (r * s - sh2) / sub[t + 1] + sup[t];
      const double v1 = dia[t + 1] - Tmm - r - s;
      const double v2 = sub[t + 2];
      const double lhs = sub[t] * (fabs(v1) + fabs(v2));
      const double rhs = v0 * (fabs(dia[t - 1]) + fabs(Tmm) + fabs(dia[t + 1]));
      hit = fabs(lhs) < eps * rhs;
    }
    const int im = max(highest(hit), il);
    {  // 12 operations for each of the iu-k+1 columns and min(iu, k+3)+1 rows of steps im..iu-2
      const int a = iu - im, m = a - 2;
      work += 12.0 * ((a + 1) * (a + 2) / 2 - 3 + m * (im + iu - 3) / 2 + 4 * m + iu + 1);
    }
    double x0, x1, x2;
    {
      const double Tmm = dia[im];
      const double r = sh0 - Tmm, s = sh1 - Tmm;
      x0 = (r * s - sh2) / sub[im + 1] + sup[im];
      x1 = dia[im + 1] - Tmm - r - s;
      x2 = sub[im + 2];
    }
    // ---- first window's rows im+3 .. im+PB+2 (slots 0..PB-1), columns im .. im+63; its open rows
    {
      const int c = im + lane, cc = min(c, iu);
      double v[PB / NW], o = 0;
#pragma unroll
      for (int j = 0; j < PB / NW; j++) v[j] = AT(min(im + 3 + wave + NW * j, iu), cc);
      if (wave < 3) o = AT(min(im + wave, iu), cc);
#pragma unroll
      for (int j = 0; j < PB / NW; j++) {
        const int r = im + 3 + wave + NW * j;
        win[0][(wave + NW * j) * PWP + lane] = c >= r ? v[j] : c == r - 1 ? sub[min(r, iu)] : 0.0;
      }
      if (wave < 3) {  // the bulge's columns: subdiagonal entries, then zeros
        if (lane < wave) o = lane == wave - 1 ? sub[im + wave] : 0.0;
        hand[0][wave][lane] = o;
      }
    }
    const int sc = im + t;  // column of a lane of waves 1-3: im + 64 + (t - 64)
    double s0 = 0, s1 = 0;  // its open rows
    if (wave > 0 && sc <= iu) {
      s0 = AT(im, sc);
      s1 = AT(im + 1, sc);
    }
    const double subim = sub[im];
    __syncthreads();
    int par = 0, wcur = 0;
    int pk0 = 0, pn = 0;  // previous window: first step, steps (0: none)
    // right updates of the previous window on rows k1-1 down to 0, PT rows per
    // item: its own rows (from its buffer), then the rows above (from global
    // memory), through the wave's transpose buffer
    auto right_items = [&](int first, int stride, bool last) {
      const SchurRf *rp = rf[par ^ 1];
      const double *wp = win[wcur == 0 ? 2 : wcur - 1];
      const unsigned fon = (unsigned)__ballot(lane < pn && rp[min(lane, PB - 1)].app != 0);
      const bool full = fon == (1u << PB) - 1;
      const int nc = pn + 2, nrow = pk0 + pn;
      double *tb = tbuf[wave];
      for (int it = first; it * PT < nrow; it += stride) {
        const int rtop = nrow - 1 - it * PT;  // row of tb's row 0; row rr holds rtop - rr
        const int nr = min(PT, rtop + 1), own = it == 0 ? pn : 0;
        int rb = lane >> 5;
        asm volatile("" : "+v"(rb));  // per-row values are formed here, not hoisted
        const int cl5 = lane & 31, cc = min(cl5, nc - 1);
#pragma unroll
        for (int h = 0; h < PT / 2; h += 16) {
          double v[16];
#pragma unroll
          for (int j = 0; j < 16; j++) v[j] = AT(max(rtop - (rb + 2 * (h + j)), 0), pk0 + cc);
          if (own && h == 0) {
#pragma unroll
            for (int j = 0; j < PB / 2; j++) {
              const int rr = rb + 2 * j;
              const double o = wp[max(pn - 1 - rr, 0) * PWP + cc];
              v[j] = rr < own ? o : v[j];
            }
          }
          if (cl5 < nc)
#pragma unroll
            for (int j = 0; j < 16; j++) tb[(rb + 2 * (h + j)) * PTP + cl5] = v[j];
        }
        wave_sync();
        if (lane < nr) {
          double *row = tb + lane * PTP;
          if (full && !own) schur_right<true>(0, rp, row);
          // a row of the window takes part from its own step on
          else schur_right<false>(own ? fon & (~0u << max(pn - 1 - lane, 0)) : fon, rp, row);
          if (last && fin[2] != 0.0) {
            const double tau = fin[0], e0 = fin[1], u0 = row[pn], u1 = row[pn + 1];
            double tt = u1 * e0;
            tt += u0;
            const double w = tau * tt;
            row[pn] = u0 - w;
            row[pn + 1] = u1 - w * e0;
          }
        }
        wave_sync();
        asm volatile("" : "+v"(rb));
        if (cl5 < nc) {
          gptr<double> g = A + ((long)(rtop - rb) * n + pk0 + cl5);
#pragma unroll
          for (int h = 0; h < PT / 2; h += 8) {
            double o[8];
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = tb[(rb + 2 * (h + j)) * PTP + cl5];
            if ((own == 0 || 2 * h >= own) && 2 * h + 16 <= nr) {
#pragma unroll
              for (int j = 0; j < 8; j++) g[-(long)(2 * (h + j)) * n] = o[j];
            } else {  // a window row stores its columns from the diagonal on
#pragma unroll
              for (int j = 0; j < 8; j++) {
                const int rr = rb + 2 * (h + j), r = rtop - rr;
                if (r >= 0 && pk0 + cl5 >= (rr < own ? r : 0)) AT(r, pk0 + cl5) = o[j];
              }
            }
          }
        }
        wave_sync();
      }
      // the window rows' columns beyond its right updates
      if (wave == NW - 1 && lane >= nc && pk0 + lane <= iu) {
        double o[PB];
#pragma unroll
        for (int j = 0; j < PB; j++) o[j] = wp[j * PWP + lane];
#pragma unroll
        for (int j = 0; j < PB; j++)
          if (j < pn) AT(pk0 + j, pk0 + lane) = o[j];
      }
    };
    // after the last window one round more applies its right updates, on all waves
    for (int k0 = im;; k0 += PB) {
      const bool chase = k0 <= iu - 2;
      const int k1 = min(k0 + PB, iu - 1), nstep = k1 - k0;
      const bool more = k1 < iu - 1;
      const int wnext = wcur == 2 ? 0 : wcur + 1;
      if (wave == 0 && chase) {
        double *W = win[wcur];
        double a0 = hand[par][0][lane], a1 = hand[par][1][lane], a2 = hand[par][2][lane];
        double nv = W[lane];
        SchurRf *R = rf[par];
        // one step with operands well inside the normal range (false: not
        // done).  q is a constant in each of the PB copies, so lanes, lane
        // masks and LDS offsets are
        const unsigned rfa = (unsigned)(uintptr_t)(__attribute__((address_space(3))) SchurRf *)R;
        const unsigned sba = (unsigned)(uintptr_t)(__attribute__((address_space(3))) double *)(sub + k0);
        auto fast = [&](auto qc) __attribute__((always_inline)) {
          constexpr int q = decltype(qc)::value;
          double least;
          __asm__("v_min_f64 %0, |%1|, |%2|" : "=v"(least) : "v"(x1), "v"(x2));
          if (__builtin_expect(__ballot(least >= 0x1p-350) == 0, 0)) return false;
          double tail = x1 * x1;
          tail += x2 * x2;
          const double sq = x0 * x0 + tail;
          double bb = root(sq, __builtin_amdgcn_rsq(sq));
          if (x0 >= 0) bb = -bb;
          const double den = x0 - bb;
          const double yd = recip(den, __builtin_amdgcn_rcp(den)), yb = recip(bb, __builtin_amdgcn_rcp(bb));
          const double e0 = quot(x1, den, yd), e1 = quot(x2, den, yd);
          const double tau = quot(-den, bb, yb);  // bb - x0 = -den exactly
          const schur_d2 o0 = {tau, e0}, o1 = {e1, __longlong_as_double((1ll << 32) | (unsigned)(base + q + 1))};
          // one lane writes the reflector, its step number last
          __asm__ volatile(
              "s_mov_b64 exec, 1\n\tds_write_b128 %0, %2 offset:%5\n\tds_write_b128 %0, %3 offset:%6\n\t"
              "ds_write_b64 %1, %4 offset:%7\n\ts_mov_b64 exec, -1"
              :
              : "v"(rfa), "v"(sba), "v"(o0), "v"(o1), "v"(bb), "n"(q * (int)sizeof(SchurRf)),
                "n"(q * (int)sizeof(SchurRf) + 16), "n"(q * 8)
              : "memory");
          double tt = e0 * a1;
          tt += e1 * a2;
          tt += a0;
          a0 -= tau * tt;
          a1 -= (tau * e0) * tt;
          a2 -= (tau * e1) * tt;
          W[q * PWP + lane] = a0;
          const double r10 = lane_value(a1, q), r11 = lane_value(a1, q + 1), r12 = lane_value(a1, q + 2);
          const double r20 = lane_value(a2, q), r21 = lane_value(a2, q + 1), r22 = lane_value(a2, q + 2);
          const double s3 = lane_value(nv, q + 2);
          tt = r11 * e0; tt += r12 * e1; tt += r10;
          const double w1 = tau * tt;
          x0 = r10 - w1;
          tt = r21 * e0; tt += r22 * e1; tt += r20;
          const double w2 = tau * tt;
          x1 = r20 - w2;
          tt = s3 * e1 + 0.0;  // (0 * e0 + s3 * e1) + 0 with e0 finite
          const double w3 = tau * tt;
          x2 = 0.0 - w3;
          // columns k+1 (factor e0) and k+2 (e1) of rows k+1..k+3, in their own lanes
          double f, m1, m2, m3;
          __asm__ volatile(
              "s_mov_b64 exec, %12\n\tv_mov_b64 %3, %10\n\ts_mov_b64 exec, %13\n\tv_mov_b64 %3, %11\n\t"
              "s_mov_b64 exec, %14\n\tv_mul_f64 %4, %7, %3\n\tv_mul_f64 %5, %8, %3\n\tv_mul_f64 %6, %9, %3\n\t"
              "v_add_f64 %0, %0, -%4\n\tv_add_f64 %1, %1, -%5\n\tv_add_f64 %2, %2, -%6\n\ts_mov_b64 exec, -1"
              : "+v"(a1), "+v"(a2), "+v"(nv), "=&v"(f), "=&v"(m1), "=&v"(m2), "=&v"(m3)
              : "v"(w1), "v"(w2), "v"(w3), "v"(e0), "v"(e1), "n"(1 << (q + 1)), "n"(1 << (q + 2)), "n"(3 << (q + 1)));
          a0 = a1;
          a1 = a2;
          a2 = nv;
          if (q + 1 < PB) nv = W[(q + 1) * PWP + lane];
          return true;
        };
        // the first vector is no entry of T: its size is checked apart
        const bool sized = __ballot(cap <= 0x1p340) && (k0 > im || __ballot(fabs(x0) <= 0x1p340 && fabs(x1) <= 0x1p340 && fabs(x2) <= 0x1p340));
        const int done = schur_steps(fast, sized ? nstep & ~3 : 0, std::make_integer_sequence<int, PB>());
        // the steps left: the last of a short window, or out-of-range operands
        for (int q = done; q < nstep; q++) {
          double tail = x1 * x1;
          tail += x2 * x2;
          double tau = 0, e0 = 0, e1 = 0, beta = x0;
          if (tail != 0.0) {
            double bb = sqrt(x0 * x0 + tail);
            if (x0 >= 0) bb = -bb;
            e0 = x1 / (x0 - bb);
            e1 = x2 / (x0 - bb);
            tau = (bb - x0) / bb;
            beta = bb;
          }
          const bool app = __ballot(beta != 0) != 0;
          if (lane == 0) {
            R[q].tau = tau;
            R[q].e0 = e0;
            R[q].e1 = e1;
            R[q].app = app;
            sub[k0 + q] = beta;
            __asm__ volatile("" ::: "memory");
            R[q].gen = base + q + 1;
          }
          double w1 = 0, w2 = 0, w3 = 0;
          if (app) {
            double tt = e0 * a1;
            tt += e1 * a2;
            tt += a0;
            a0 -= tau * tt;
            a1 -= (tau * e0) * tt;
            a2 -= (tau * e1) * tt;
          }
          W[q * PWP + lane] = a0;
          x0 = lane_value(a1, q);
          x1 = lane_value(a2, q);
          x2 = 0.0;
          if (app) {
            double tt = lane_value(a1, q + 1) * e0;
            tt += lane_value(a1, q + 2) * e1;
            tt += x0;
            w1 = tau * tt;
            tt = lane_value(a2, q + 1) * e0;
            tt += lane_value(a2, q + 2) * e1;
            tt += x1;
            w2 = tau * tt;
            tt = 0.0 * e0;
            tt += lane_value(nv, q + 2) * e1;
            tt += 0.0;
            w3 = tau * tt;
            x0 -= w1;
            x1 -= w2;
            x2 -= w3;
            const double f = lane == q + 1 ? e0 : e1;
            if (lane == q + 1 || lane == q + 2) {
              a1 -= w1 * f;
              a2 -= w2 * f;
              nv -= w3 * f;
            }
          }
          a0 = a1;
          a1 = a2;
          a2 = nv;
          if (q + 1 < PB) nv = W[(q + 1) * PWP + lane];
        }
        if (lane == 0 && k0 == im)  // T(im, im-1): negated where the first reflector applies above il
          sub[im] = im > il && rf[par][0].app ? -subim : subim;
        if (more) {
          if (lane >= PB) {
            hand[par ^ 1][0][lane - PB] = a0;
            hand[par ^ 1][1][lane - PB] = a1;
            hand[par ^ 1][2][lane - PB] = a2;
          }
        } else {  // the last reflector: rows iu-1, iu, columns iu-1, iu
          double p00 = lane_value(a0, nstep), p01 = lane_value(a0, nstep + 1);
          double p10 = lane_value(a1, nstep), p11 = lane_value(a1, nstep + 1);
          double tail = 0;
          tail += x1 * x1;
          double tau = 0, e0 = 0, beta = x0;
          if (tail != 0.0) {
            double bb = sqrt(x0 * x0 + tail);
            if (x0 >= 0) bb = -bb;
            e0 = x1 / (x0 - bb);
            tau = (bb - x0) / bb;
            beta = bb;
          }
          const bool app = beta != 0;
          if (app) {
            const double f0 = tau * e0;
            double tt = e0 * p10; tt += p00;
            p00 -= tau * tt; p10 -= f0 * tt;
            tt = e0 * p11; tt += p01;
            p01 -= tau * tt; p11 -= f0 * tt;
            tt = p01 * e0; tt += p00;
            double w = tau * tt;
            p00 -= w; p01 -= w * e0;
            tt = p11 * e0; tt += p10;
            w = tau * tt;
            p10 -= w; p11 -= w * e0;
            work += 6.0 * (2 + iu + 1);
          }
          if (lane == 0) {
            sub[iu - 1] = beta;
            sub[iu] = p10;
            AT(iu - 1, iu - 1) = p00;
            AT(iu - 1, iu) = p01;
            AT(iu, iu) = p11;
            fin[0] = tau;
            fin[1] = e0;
            fin[2] = app ? 1.0 : 0.0;
          }
        }
      } else {
        const int cE = k0 + 64;  // first column right of the band
        const bool act = sc >= cE && sc <= iu;
        // the window's rows of this lane's column, and the next window's rows, in flight
        constexpr int NX = (PB + NW - 1) / (NW - 1);  // PB + 1 rows over the NW - 1 waves
        double w[PB], nx[NX];
        const int c2 = k1 + lane, cc2 = min(c2, iu), ccol = min(sc, iu);
        if (more) {
#pragma unroll
          for (int q = 0; q < PB; q++) w[q] = AT(min(k0 + 2 + q, iu), ccol);
#pragma unroll
          for (int j = 0; j < NX; j++) nx[j] = AT(min(k1 + 2 + wave - 1 + (NW - 1) * j, iu), cc2);
        }
        __builtin_amdgcn_sched_barrier(0);
        // waves 5-7, which have no columns of the left strip, come first, and
        // wave 4, which shares its SIMD with the chase, last
        if (pn) {
          const int first = !chase ? wave : NW == 4 ? wave - 1 : wave > 4 ? wave - 5 : wave + 2;
          right_items(first, chase ? NW - 1 : NW, !chase);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
#pragma unroll
          for (int j = 0; j < NX; j++) {
            const int i = wave - 1 + (NW - 1) * j;  // row k1 + 2 + i
            if (i == 0) {
              if (c2 >= cE) hand[par ^ 1][2][lane] = nx[j];
            } else if (i <= PB) {
              const int r = k1 + 2 + i;
              win[wnext][(i - 1) * PWP + lane] = c2 >= r ? nx[j] : c2 == r - 1 ? sub[min(r, iu)] : 0.0;
            }
          }
          if (__ballot(act) != 0) {
            const SchurRf *R = rf[par];
            // wave 0 publishes every step of its window, within microseconds.
            // Should it not, the sweeps end all the same (their number is
            // limited), on what lies in LDS, and k_har_final finds the mark and
            // fails the call.  What the mark is and where it is set decide which
            // registers the compiler spills: so, either launch takes 0.7 to 1% more
            // than without one; with the other's, 1.4 and 1.5%.
            auto lose = [&] {
              if (NW == 8) H.count[angle] = -1;
              else const_cast<int *>(order)[gridDim.y + ORDER_LOST] = 1;
            };
            auto await = [&](int q) {
              int spin = 0;
              for (; NW == 8 || spin < POLLS; spin++) {
                if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(&R[q].gen, __ATOMIC_RELAXED,
                                                                     __HIP_MEMORY_SCOPE_WORKGROUP)) == base + q + 1)
                  break;
                if (NW == 8 && spin == POLLS) {
                  lose();
                  break;
                }
                __builtin_amdgcn_s_sleep(1);
              }
              if (NW == 4 && __builtin_expect(spin == POLLS, 0)) lose();
              __asm__ volatile("" ::: "memory");
            };
#pragma unroll
            for (int q = 0; q < PB; q++) {
              if (q % 4 == 0) await(q + 3);  // four steps at a time
              const double tau = R[q].tau, e0 = R[q].e0, e1 = R[q].e1;
              double u2 = w[q];
              if (__builtin_amdgcn_readfirstlane(R[q].app)) {
                double tt = e0 * s1;
                tt += e1 * u2;
                tt += s0;
                s0 -= tau * tt;
                s1 -= (tau * e0) * tt;
                u2 -= (tau * e1) * tt;
              }
              if (act) AT(k0 + q, sc) = s0;
              s0 = s1;
              s1 = u2;
            }
            if (act && sc < cE + PB) {
              hand[par ^ 1][0][sc - k1] = s0;
              hand[par ^ 1][1][sc - k1] = s1;
            }
          }
        }
      }
      if (!chase) break;
      __syncthreads();
      base += nstep;
      pk0 = k0;
      pn = nstep;
      par ^= 1;
      wcur = wnext;
    }
    reload = true;
  }
  __syncthreads();
  // eigenvalue 2 in Schur-diagonal order (EigenSolver::compute, EigenSolver.h:364-381)
  if (t == 0) {
    double f = 0.0;
    if (n >= 3) {
      int i = 0;
      double re2 = 0, im2 = 0;
      while (i < n && i <= 2) {
        if (i == n - 1 || sub[i + 1] == 0) {
          if (i == 2) { re2 = AT(i, i); im2 = 0; }
          ++i;
        } else {
          const double p = 0.5 * (AT(i, i) - AT(i + 1, i + 1));
          const double z = sqrt(fabs(p * p + sub[i + 1] * AT(i, i + 1)));
          if (i == 2) { re2 = AT(i + 1, i + 1) + p; im2 = z; }
          if (i + 1 == 2) { re2 = AT(i + 1, i + 1) + p; im2 = -z; }
          i += 2;
        }
      }
      f = (im2 == 0) ? sqrt(re2) : 0.0;
    }
    H.feat[angle * 14 + 13] = f;
    H.work[angle] = work;
  }
#undef AT
}

// mean and range over the 4 angles, reference output order (haralick.cpp:96-143)
// *lost: a wave of k_har_schur waited in vain
__global__ void k_har_final(const HarDesc *hd, const int *order, OutRef o, int *lost) {
  const HarDesc H = hd[blockIdx.x];
  if (threadIdx.x != 0) return;
  bool hit = order[gridDim.x + ORDER_LOST] != 0;
  for (int g = 0; g < 4; g++) hit |= H.count[g] < 0;
  if (hit) __hip_atomic_store(lost, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  double temp[28];
  for (int a = 0; a < 14; a++) {
    double s = 0, mn = kInf, mx = -kInf;
    for (int g = 0; g < 4; g++) {
      const double v = H.feat[g * 14 + a];
      s += v;
      if (v < mn) mn = v;
      if (v > mx) mx = v;
    }
    temp[a] = s / 4;
    temp[a + 14] = mx - mn;
  }
  const int ord[28] = {0, 14, 1, 15, 2, 16, 9, 23, 10, 24, 8, 22, 11, 25,
                       4, 18, 13, 27, 12, 26, 5, 19, 7, 21, 6, 20, 3, 17};
  double *out = o.rows[blockIdx.x];
  for (int a = 0; a < 28; a++) out[a] = temp[ord[a]];
}

void launch_haralick_prep(const Img *imgs, const Stats *st, const HarDesc *hd, int nimg, int maxn, hipStream_t s) {
  int blocks = (maxn + 255) / 256;
  if (blocks > 1024) blocks = 1024;
  k_har_quant<<<dim3(blocks, nimg), 256, 0, s>>>(imgs, st, hd);
  k_har_lut<<<nimg, 64, 0, s>>>(hd);
  static const bool lds_ok = hipFuncSetAttribute((const void *)k_har_cooc, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                  256 * 257 / 2 * sizeof(uint32_t)) == hipSuccess;
  (void)lds_ok;
  k_har_cooc<<<dim3(4, nimg), 1024, 256 * 257 / 2 * sizeof(uint32_t), s>>>(imgs, hd);
  k_har_stats<<<dim3(4, nimg), 256, 0, s>>>(hd);
  k_har_q<<<xcd_grid(QRB, 4 * nimg), 256, 0, s>>>(hd, nimg);
}
// Entries in decreasing order of tones (ng), for the eigen kernels: their
// cost grows with ng (about ng^2 for the Schur sweeps, ng^3 for the
// Hessenberg reduction), and ng ranges over 10..256 within a batch, so
// dispatching the largest matrices first keeps the last wave of blocks
// short (longest processing time first).  Every matrix is computed on its
// own, so the order changes no result.  Thread b owns key b = 256 - ng and
// scans the entries in index order (keys staged in LDS, chunk by chunk), so
// ties keep index order and the order is the same on every run.
//
// order[nimg + ORDER_PICK] (pick_too) tells which kernel finishes a launch of medium size
// (launch_haralick_qr): 1 for k_har_schur<4>, whose 512 resident matrices make
// short chains, 0 for k_har_qr, whose 4,096 make three times longer ones but do
// 1.1 to 2.5 times as many matrices in all.  The estimates, in ms, follow either
// kernel's times over 95 launches of 1,056 to 6,000 matrices: equal tones (8 ..
// 240), tones spread evenly or thinly from 0, two kinds of them, one entry in 40 of
// 256 tones, and nodes of images.  There the choice is the slower kernel by 2% at
// most where that is k_har_schur, by 5% where it is k_har_qr.
// Either kernel gives the same bits.
constexpr int ORDER_CHUNK = 16384;
__global__ void __launch_bounds__(320) k_har_order(const int *ng, int nimg, int *order, int pick_too) {
  __shared__ __align__(16) uint16_t key[ORDER_CHUNK];
  __shared__ int cnt[257];
  __shared__ double shd[5];
  const int t = threadIdx.x;
  for (int b = t; b < 257; b += blockDim.x) cnt[b] = 0;
  __syncthreads();
  for (int e = t; e < nimg; e += blockDim.x) atomicAdd(&cnt[256 - min(max(ng[e], 0), 256)], 1);
  __syncthreads();
  if (t == 0) {
    int sum = 0;
    for (int b = 0; b < 257; b++) {
      const int c = cnt[b];
      cnt[b] = sum;
      sum += c;
    }
  }
  __syncthreads();
  if (pick_too) {
    const double n = 256 - t, m = t < 257 ? 4.0 * ((t < 256 ? cnt[t + 1] : nimg) - cnt[t]) : 0.0;
    const double chain = n * (8.1e-3 + n * (2.05e-4 + n * 1.5e-7));  // one matrix by k_har_schur<4>
    // its matrices from the largest to order n need so many rounds of 512, none shorter
    const double rounds = m > 0 ? ceil((t < 256 ? cnt[t + 1] : nimg) / 128.0) * chain : 0.0;
    const double longest = block_reduce(rounds, MaxOp(), shd);
    const double chains = block_reduce(m * chain, SumOp(), shd);
    const double top = block_reduce(m > 0 ? n : 0.0, MaxOp(), shd);
    const double work = block_reduce(m * n * n * (1.5e-7 + n * 7.6e-10), SumOp(), shd);
    if (t == 0) {
      const double schur = fmax(longest, chains / 512);
      const double qr = top * (3e-3 + top * (5.4e-4 + top * 8.1e-7)) + 0.42 * work;
      order[nimg + ORDER_PICK] = schur < qr;
    }
  }
  if (t == 0) {  // cnt[256 - n]: entries of more than n tones
    const int end = cnt[256 - 2], large = cnt[256 - HESS_SMALL];
    order[nimg + ORDER_END] = end;
    order[nimg + ORDER_LOST] = 0;
    order[nimg + ORDER_LARGE] = end - large >= HESS_MANY ? large : end;
  }
  int pos = t < 257 ? cnt[t] : 0;
  for (int base = 0; base < nimg; base += ORDER_CHUNK) {
    const int m = min(ORDER_CHUNK, nimg - base), m8 = (m + 7) & ~7;
    __syncthreads();  // the previous chunk's keys are consumed
    for (int e = t; e < m8; e += blockDim.x)  // pad to eight keys with a key no thread owns
      key[e] = e < m ? (uint16_t)(256 - min(max(ng[base + e], 0), 256)) : (uint16_t)0xffff;
    __syncthreads();
    if (t < 257)
      for (int e = 0; e < m8; e += 8) {  // eight keys per LDS read
        const uint4 kk = *(const uint4 *)(key + e);
        const unsigned w[4] = {kk.x, kk.y, kk.z, kk.w};
#pragma unroll
        for (int j = 0; j < 8; j++)
          if ((int)((w[j >> 1] >> (16 * (j & 1))) & 0xffff) == t) order[pos++] = base + e + j;
      }
  }
}
// Matrices of a launch that k_har_order picks the kernel for.
static bool haralick_pick(int nimg) { return 4 * nimg > 1024 && 4 * nimg <= 6144; }
void launch_haralick_order(const int *ng, int nimg, int *order, hipStream_t s) {
  k_har_order<<<1, 320, 0, s>>>(ng, nimg, order, haralick_pick(nimg));
}
void launch_haralick_hess(const HarDesc *hd, const int *order, int nimg, hipStream_t s) {
  k_har_hess<8, 256><<<dim3(4, nimg), 512, 0, s>>>(hd, order);
  if (nimg >= HESS_MANY) k_har_hess<1, HESS_SMALL><<<dim3(4, nimg), 64, 0, s>>>(hd, order);
  k_har_hess_rows<<<dim3(4, nimg, (256 - 2 + RWS - 1) / RWS), 64, 0, s>>>(hd, order);
}
void launch_haralick_qr(const HarDesc *hd, const int *order, bool no_polls, int nimg, hipStream_t s) {
  // Up to 256 matrices every CU has at most one, and the launch lasts as long
  // as the longest chain of steps: eight waves per matrix.  Up to 1024, four
  // waves per matrix, two matrices per CU: with tones of 8 .. 240, equal or
  // spread, in no case slower than the kernel before it (240 equal tones, 1024
  // matrices: 37.3 against 72.4 ms; 64: 2.9 against 5.7; 8: 0.18 against 0.19).
  // Beyond 6144 one wave per matrix and sixteen matrices per CU: its chain is
  // three times slower, but it does less work per step, and with that many the
  // work counts.  Between, it depends on the tones, which only the device knows:
  // 1600 matrices of 64 equal tones 5.4 ms by four waves and 3.4 by one, of 0 ..
  // 253 tones 21.6 and 49.9.  Both are launched and one of them returns at once.
  // Nodes of 256 x 256 images (tones 10..256, mean 128): 48 matrices 12.5 ms (30.6
  // with one 256-thread block per matrix; four waves: 17.5), 1200 18.5 against
  // 47.4, 2400 33.3 against 51.1, 4800 63.1 against 69.2; 7200 87.7 by one wave
  // against 93.9, 9600 112.0 against 124.8, 19200 200 against 259.
  const dim3 grid(4, nimg);
  const int *pick = haralick_pick(nimg) ? order + nimg + ORDER_PICK : nullptr;
  if (no_polls && 4 * nimg <= 256) k_har_schur<8, 0><<<grid, 512, 0, s>>>(hd, order, nullptr);
  else if (no_polls) k_har_schur<4, 0><<<grid, 256, 0, s>>>(hd, order, nullptr);
  else if (4 * nimg <= 256) k_har_schur<8><<<grid, 512, 0, s>>>(hd, order, nullptr);
  else if (4 * nimg <= 6144) k_har_schur<4><<<grid, 256, 0, s>>>(hd, order, pick);
  if (!no_polls && (pick || 4 * nimg > 6144)) k_har_qr<<<grid, 64, 0, s>>>(hd, order, pick);
}
void launch_haralick_final(const HarDesc *hd, const int *order, OutRef o, int *lost, int nimg, hipStream_t s) {
  k_har_final<<<nimg, 64, 0, s>>>(hd, order, o, lost);
}

// ======================================================================= Tamura
// tamura.cpp:10-299.  The scratch's layout is given at tam_summary.
// (x - min) / max per pixel; planes are 256-byte aligned (arena), so each
// thread streams two double pairs through the global address space
typedef double tam_d2 __attribute__((ext_vector_type(2)));
__global__ void __launch_bounds__(256) k_tam_norm(const Img *imgs, const Stats *st, double *const *scr) {
  const Img im = imgs[blockIdx.y];
  const Stats S = st[blockIdx.y];
  const long n = (long)im.h * im.w, n4 = n >> 2;
  const gptr<const tam_d2> src = (gptr<const tam_d2>)to_global((const double *)im.p);
  const gptr<tam_d2> dst = (gptr<tam_d2>)to_global(scr[blockIdx.y]);
  const double mn = S.mn, mx = S.mx;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n4; i += (long)gridDim.x * blockDim.x) {
    tam_d2 a = src[2 * i], b = src[2 * i + 1];
    a.x = (a.x - mn) / mx;
    a.y = (a.y - mn) / mx;
    b.x = (b.x - mn) / mx;
    b.y = (b.y - mn) / mx;
    dst[2 * i] = a;
    dst[2 * i + 1] = b;
  }
  if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
    const long i = (n4 << 2) + threadIdx.x;
    scr[blockIdx.y][i] = (im.p[i] - mn) / mx;
  }
}

// the value of the lane below (lane - 1); lane 0 takes `first`
__device__ __forceinline__ double from_lane_below(double v, double first) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(first), __double2loint(v), 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(first), __double2hiint(v), 0x138, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// Sums over a plane that the directionality and contrast need, by wave of
// k_tam_pix (64 columns x tam_rows rows), then by block of TAM_CHUNK pixels
struct TamPart { double s, sr, pmn, pmx; int ks, kmask; };
struct TamPart2 { double m2, m4; };
struct TamSum { double mean, sr, pmn, pmx; long long ks; int kmn, kmx; int hk[3], hd[125]; };
constexpr int TAM_CHUNK = 16384;
static_assert(sizeof(TamPart) % 8 == 0 && sizeof(TamPart2) % 8 == 0, "parts are laid out in doubles");
// scratch of a plane of P pixels, in doubles: [0, P) normalised plane, [P, 2P)
// row differences and [3P, 4P) corner differences of the summed-area table,
// [2P, 3P) phi, [4P, 4.5P) best scale (int), then the summary, the parts of
// k_tam_pix and of k_tam_hist and a row of the table
__host__ __device__ inline size_t tam_summary(long P) { return 4 * (size_t)P + ((size_t)P + 1) / 2; }
__host__ __device__ inline size_t tam_parts(long P) { return tam_summary(P) + (sizeof(TamSum) + 7) / 8; }
// rows of a wave of k_tam_pix: eight reuse what neighbouring rows share, two make
// the shorter chain where a plane has few waves (one of 64 x 64: 10.5 us, 29.3 by eight)
__host__ __device__ inline int tam_rows(int h, int w) { return (long)h * w <= 4096 ? 2 : 8; }
__host__ __device__ inline int tam_runs(int h, int w) { return ((w + 63) / 64) * ((h + tam_rows(h, w) - 1) / tam_rows(h, w)); }
__host__ __device__ inline size_t tam_parts2(int h, int w) {
  return tam_parts((long)h * w) + (size_t)tam_runs(h, w) * (sizeof(TamPart) / 8);
}
__host__ __device__ inline size_t tam_row(int h, int w) {
  return tam_parts2(h, w) + ((size_t)h * w + TAM_CHUNK - 1) / TAM_CHUNK * (sizeof(TamPart2) / 8);
}
size_t tamura_scratch(int h, int w) { return tam_row(h, w) + w + 8; }
// the most waves that a plane of up to maxh x maxw pixels has: more rows make
// more of them until a plane takes eight rows per wave
static int tam_max_runs(int maxh, int maxw) {
  int most = tam_runs(maxh, maxw);
  for (int w = 16; w <= maxw; w = (w + 63) / 64 * 64 + 1)  // the narrowest of each number of columns of waves
    most = std::max(most, tam_runs(std::min(maxh, std::max(4096 / w, 1)), w));
  return most;
}

// Summed-area table with the reference's exact recurrence
//   S(y,x) = ((I(y,x) + S(y,x-1)) + S(y-1,x)) - S(y-1,x-1)
// and from it what k_tam_pix reads: R = S(y,x) - S(y,x-1) and
// D = S(y,x) - S(y,x-1) - S(y-1,x) + S(y-1,x-1), with zeros outside the plane.
//
// An anti-diagonal wavefront: lane l of a wave owns row y0 + l of a 64-row
// strip and is l columns behind lane 0; the value above comes from lane l - 1.
// The chain is three additions and a lane shift per step, so a plane's strips
// run at once: strip s belongs to wave s % nw and starts LAG = 5 groups of 16
// steps behind strip s - 1, whose last row it takes from a ring of 64 values.
// A wave's next strip begins T groups after its last, T >= 5 nw + 1, and what
// wave 0 takes from the strip before it passes through a row in memory.  A
// group's 64 x 16 inputs and results pass through an LDS tile, so that 16 lanes
// access 128 consecutive bytes of a row.  A block has as many waves, and LDS, as
// the highest plane has strips (2,000 planes of 16 x 16: 20 us, 47 with LDS for
// eight).  Three planes of 1388 x 1040 and their
// transforms (18 planes): 1.2 ms, 9.0 ms with one wave per plane that met at
// two barriers per step; 4,800 planes of up to 256 x 256 (7.6 GB moved): 3.0 ms.
constexpr int SAT_WAVES = 8, SAT_GR = 16, SAT_TILE = 64 * (SAT_GR + 1);
__global__ void __launch_bounds__(64 * SAT_WAVES) k_tam_sat(const Img *imgs, double *const *scr) {
  constexpr int GR = SAT_GR, LAG = 5;
  extern __shared__ double sat_lds[];  // a tile and a ring per wave
  double (*const tiles)[SAT_TILE] = (double (*)[SAT_TILE])sat_lds;
  double (*const rings)[64] = (double (*)[64])(sat_lds + (blockDim.x >> 6) * SAT_TILE);
  const Img im = imgs[blockIdx.x];
  const int H = im.h, W = im.w;
  const long P = (long)H * W;
  const gptr<double> N = to_global(scr[blockIdx.x]);
  const gptr<const double> I = (gptr<const double>)N;
  const gptr<double> R = N + P, D = N + 3 * P, last = N + tam_row(H, W);
  const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  double *const tile = tiles[w], *const ring = rings[w];  // ring: the row above this wave's strip
  double *const below = rings[w + 1 < nw ? w + 1 : 0];
  const int G = (W + 63 + GR - 1) / GR, T = max(G, LAG * nw + 1);
  const int strips = (H + 63) / 64;
  const int rounds = (strips - 1) / nw * T + LAG * ((strips - 1) % nw) + G;
  const int lr = l >> 4, lc = l & 15;
  double nx[GR], nup = 0.0;
  // inputs of group g of strip st (and of the row above, where it is in memory)
  auto fetch = [&](int st, int g) {
    const int y0 = st * 64;
#pragma unroll
    for (int k = 0; k < GR; k++) {
      const int r = 4 * k + lr, y = y0 + r, x = g * GR - r + lc;
      nx[k] = (y < H && (unsigned)x < (unsigned)W) ? I[(long)y * W + x] : 0.0;
    }
    if (w == 0) {
      const int x = g * GR + lc;
      nup = (st > 0 && x < W) ? last[x] : 0.0;
    }
  };
  double cur = 0, up_prev = 0;
  for (int r = 0; r < rounds; r++) {
    const int q = r - LAG * w;             // rounds since this wave's first strip began
    const int pass = q >= 0 ? q / T : 0, g = q - pass * T;
    const int st = pass * nw + w;
    if (q >= 0 && g < G && st < strips) {  // uniform over the wave
      if (g == 0) {
        fetch(st, 0);
        cur = up_prev = 0;
      }
#pragma unroll
      for (int k = 0; k < GR; k++) tile[(4 * k + lr) * (GR + 1) + lc] = nx[k];
      if (w == 0 && l < GR) ring[(q * GR + l) & 63] = nup;
      if (g + 1 < G) fetch(st, g + 1);     // in flight during this group
      wave_sync();
      double v[GR], up0[GR], d[GR];
#pragma unroll
      for (int k = 0; k < GR; k++) {
        v[k] = tile[l * (GR + 1) + k];
        up0[k] = ring[(q * GR + k) & 63];
      }
      wave_sync();
#pragma unroll
      for (int k = 0; k < GR; k++) {       // columns left of the plane stay zero, those right of it are not stored
        const double up = from_lane_below(cur, up0[k]);
        const double s = v[k] + cur + up - up_prev;
        v[k] = s;
        d[k] = s - cur;
        tile[l * (GR + 1) + k] = d[k];
        d[k] = d[k] - up + up_prev;
        cur = s;
        up_prev = up;
      }
      if (l == 63) {                       // the strip's last row, by the round: a wave's strips follow on
        if (w + 1 < nw) {
#pragma unroll
          for (int k = 0; k < GR; k++) below[(q * GR + k - 63) & 63] = v[k];
        } else if (st + 1 < strips) {
#pragma unroll
          for (int k = 0; k < GR; k++) {
            const int x = g * GR + k - 63;
            if ((unsigned)x < (unsigned)W) last[x] = v[k];
          }
        }
      }
      auto store = [&](gptr<double> to) {
        wave_sync();
#pragma unroll
        for (int k = 0; k < GR; k++) {
          const int rr = 4 * k + lr, y = st * 64 + rr, x = g * GR - rr + lc;
          const double o = tile[rr * (GR + 1) + lc];
          if (y < H && (unsigned)x < (unsigned)W) to[(long)y * W + x] = o;
        }
        wave_sync();
      };
      store(R);
#pragma unroll
      for (int k = 0; k < GR; k++) tile[l * (GR + 1) + k] = d[k];
      store(D);
    }
    __syncthreads();
  }
}

// |a0 / c0 - a1 / c1| for whole numbers c <= 2^14 and r within a few units in
// the last place of 1 / c.  A quotient is the product with r with the
// remainder's quotient added, which rounds as the division does because a / c is
// nowhere nearer than 1 / (2c) units in the last place to the middle between two
// doubles.  Not so where the quotient is subnormal, which can lie in the very
// middle, or where a is infinite and the remainder no number: these are divided.
__device__ __forceinline__ double mean_diff(double a0, double c0, double r0, double a1, double c1, double r1) {
  constexpr int ODD = 0x3 | 0x10 | 0x80;  // for v_cmp_class: NaN, subnormal of either sign
  const double q0 = a0 * r0, q1 = a1 * r1;
  const double m0 = __builtin_fma(__builtin_fma(-c0, q0, a0), r0, q0);
  const double m1 = __builtin_fma(__builtin_fma(-c1, q1, a1), r1, q1);
  double v = fabs(m0 - m1);
  if (__any(__builtin_amdgcn_class(m0, ODD) || __builtin_amdgcn_class(m1, ODD))) v = fabs(a0 / c0 - a1 / c1);
  return v;
}

// Coarseness per pixel (best scale), directionality phi and the sums.
//
// The reference's window mean (efficientLocalMean, tamura.cpp) takes its four
// table entries from two adjacent rows and columns: stop row and the row above,
// start column and the one to its left.  Its numerator is thus an entry of D at
// (stop row, start column), of R where the window starts in row 0: one load.
// Its divisor is full, a power of two, away from the borders.
//
// Bound by instruction issue, so a wave takes 64 columns and goes down tam_rows
// rows: what depends on the row alone is scalar, and the rows' neighbours stay in
// registers.  4,800 planes of up to 256 x 256: 10.4 ms; 18.0 ms with four table
// entries per mean, 12.9 ms with one thread per pixel.
__global__ void __launch_bounds__(256, 3) k_tam_pix(const Img *imgs, double *const *scr, int nimg, int per_img) {
  __shared__ double recip[129];
  int ent, blk;
  if (!xcd_item(per_img, nimg, ent, blk)) return;  // one plane's tables stay in one L2
  if (threadIdx.x < 129) recip[threadIdx.x] = 1.0 / threadIdx.x;
  __syncthreads();
  const Img im = imgs[ent];
  const int H = im.h, W = im.w;
  const long P = (long)H * W;
  const int run = __builtin_amdgcn_readfirstlane(blk * 4 + (threadIdx.x >> 6));
  if (run >= tam_runs(H, W)) return;
  const int rows = tam_rows(H, W), nc = (W + 63) / 64, y0 = run / nc * rows, x0 = run % nc * 64 + (threadIdx.x & 63);
  const bool own = x0 < W;
  const int x = min(x0, W - 1);
  const gptr<double> N = to_global(scr[ent]);  // global, not FLAT: vector-memory waits only
  const gptr<const double> Nc = (gptr<const double>)N, R = Nc + P, D = Nc + 3 * P;
  const double ctl = x, ctr = W - x;  // widths of the windows beside it where the border cuts them
  const double rtl = recip[min(x, 128)], rtr = recip[min(W - x, 128)];
  const bool xm = x >= 1, xp = x + 1 < W;
  const unsigned xl = max(x - 1, 0), xr = min(x + 1, W - 1);
  // rows y - 1 and y of the normalised plane around column x
  double a0 = 0, a1 = 0, a2 = 0, b0, b1, b2;
  if (y0 >= 1) {
    const gptr<const double> q = Nc + (long)(y0 - 1) * W;
    a0 = xm ? q[xl] : 0.0;
    a1 = q[(unsigned)x];
    a2 = xp ? q[xr] : 0.0;
  }
  {
    const gptr<const double> q = Nc + (long)y0 * W;
    b0 = xm ? q[xl] : 0.0;
    b1 = q[(unsigned)x];
    b2 = xp ? q[xr] : 0.0;
  }
  TamPart T = {0, 0, 1e308, -1e308, 0, 0};
#pragma unroll 1
  for (int y = y0; y < min(y0 + rows, H); y++) {
    int xi = x;
    __asm__ volatile("" : "+v"(xi));  // formed anew per row: registers held through the loop cost more waves
    // coarseness: argmax over scales of E_h / E_v (tamura.cpp:183-238); the four
    // windows of each scale, all loads in flight
    double d[7][4], c0 = 0, c1 = 0, c2 = 0;
#pragma unroll
    for (int k = 0; k < 7; k++) {
      const int k2 = 1 << k;
      const gptr<const double> h = (y <= k2 ? R : D) + (long)min(y + k2 - 1, H - 1) * W;
      const gptr<const double> v0 = D + (long)min(y + 2 * k2 - 1, H - 1) * W;  // y >= k2: starts in row y
      const gptr<const double> v1 = (y <= 2 * k2 ? R : D) + (long)max(y - 1, 0) * W;
      d[k][0] = h[(unsigned)xi];
      d[k][1] = h[(unsigned)max(xi - 2 * k2, 0)];
      d[k][2] = v0[(unsigned)max(xi - k2, 0)];
      d[k][3] = v1[(unsigned)max(xi - k2, 0)];
    }
    if (y + 1 < H) {
      const gptr<const double> q = Nc + (long)(y + 1) * W;
      c0 = xm ? q[xl] : 0.0;
      c1 = q[(unsigned)xi];
      c2 = xp ? q[xr] : 0.0;
    }
    double maxE = 0;
    int maxk = 0;
#pragma unroll
    for (int k = 0; k < 7; k++) {
      const int k2 = 1 << k;
      const double full = 1.0 / (4 * k2 * k2);  // a power of two: the product is the quotient
      const bool okh = xi + k2 < W && xi - k2 >= 0;
      double eh = 0, ev = 0;
      if (__any(okh)) {
        const int n = min(y + k2, H) - max(y - k2, 0);
        const bool cl = xi < 2 * k2, cr = W - xi < 2 * k2;
        if (n == 2 * k2 && !__any(okh && (cl || cr))) {
          eh = fabs(d[k][0] * full - d[k][1] * full);
        } else {
          const double r = recip[n], c = n;
          eh = mean_diff(d[k][0], c * (cr ? ctr : 2.0 * k2), r * (cr ? rtr : 0.5 / k2), d[k][1],
                         c * (cl ? ctl : 2.0 * k2), r * (cl ? rtl : 0.5 / k2));
        }
        eh = okh ? eh : 0.0;
      }
      if (y + k2 < H && y - k2 >= 0) {
        const int n0 = min(2 * k2, H - y), n1 = min(2 * k2, y), wc = min(xi + k2, W) - max(xi - k2, 0);
        if (n0 == 2 * k2 && n1 == 2 * k2 && __all(wc == 2 * k2)) {
          ev = fabs(d[k][2] * full - d[k][3] * full);
        } else {
          const double r = recip[wc], c = wc;
          ev = mean_diff(d[k][2], n0 * c, recip[n0] * r, d[k][3], n1 * c, recip[n1] * r);
        }
      }
      if (eh > maxE) { maxE = eh; maxk = k + 1; }
      if (ev > maxE) { maxE = ev; maxk = k + 1; }
    }
    // directionality filters after the reference's assignments (tamura.cpp:50-57):
    // H = [-1 2 1; -2 0 2; -1 -2 -1], V = [1 0 0; 0 0 0; -1 0 0], correlation order
    // (column offset outer, row offset inner), zero weights skipped (exact); what
    // lies outside the plane is zero, and adding it changes nothing
    double dh = 0.0, dv = 0.0;
    dh += -1 * a0;
    dh += -2 * b0;
    dh += -1 * c0;
    dh += 2 * a1;
    dh += -2 * c1;
    dh += 1 * a2;
    dh += 2 * b2;
    dh += -1 * c2;
    dv += 1 * a0;
    dv += -1 * c0;
    double ph = 0.0;
    if (dh >= 0.0001) ph = atan(dv / dh) + (M_PI / 2.0 + 0.001);
    if (own) {
      const unsigned i = (unsigned)y * (unsigned)W + (unsigned)x;
      ((gptr<int>)(N + 4 * P))[i] = maxk;
      (N + 2 * P)[i] = ph;
      T.s += b1;
      if (dh >= 0.0001) T.sr += (dh * dh + dv * dv) + ph * ph;
      T.ks += maxk;
    }
    T.kmask |= 1 << maxk;
    T.pmn = fmin(T.pmn, ph);
    T.pmx = fmax(T.pmx, ph);
    a0 = b0; a1 = b1; a2 = b2;
    b0 = c0; b1 = c1; b2 = c2;
  }
  for (int o = 32; o > 0; o >>= 1) {
    T.s += __shfl_down(T.s, o, 64);
    T.sr += __shfl_down(T.sr, o, 64);
    T.pmn = fmin(T.pmn, __shfl_down(T.pmn, o, 64));
    T.pmx = fmax(T.pmx, __shfl_down(T.pmx, o, 64));
    T.ks += __shfl_down(T.ks, o, 64);
    T.kmask |= __shfl_down(T.kmask, o, 64);
  }
  if ((threadIdx.x & 63) == 0) ((TamPart *)(scr[ent] + tam_parts(P)))[run] = T;
}

// The plane's sums from its parts; clears the histograms.  By one block of 256.
__device__ __forceinline__ void tam_mid(const Img &im, const double *scr, TamSum &T) {
  __shared__ double shd[4];
  __shared__ long long shl[4];
  __shared__ int shi[4];
  const long P = (long)im.h * im.w;
  const TamPart *part = (const TamPart *)(scr + tam_parts(P));
  double s = 0, sr = 0, pmn = 1e308, pmx = -1e308;
  long long ks = 0;
  int km = 0;
  for (int b = threadIdx.x; b < tam_runs(im.h, im.w); b += 256) {
    const TamPart q = part[b];
    s += q.s;
    sr += q.sr;
    pmn = fmin(pmn, q.pmn);
    pmx = fmax(pmx, q.pmx);
    ks += q.ks;
    km |= q.kmask;
  }
  s = block_reduce(s, SumOp(), shd);
  sr = block_reduce(sr, SumOp(), shd);
  pmn = block_reduce(pmn, MinOp(), shd);
  pmx = block_reduce(pmx, MaxOp(), shd);
  ks = block_reduce(ks, SumOp(), shl);
  const int kmn = block_reduce(km ? __builtin_ctz(km) : 99, MinOp(), shi);
  const int kmx = block_reduce(km ? 31 - __builtin_clz(km) : -1, MaxOp(), shi);
  if (threadIdx.x < 125) T.hd[threadIdx.x] = 0;
  if (threadIdx.x < 3) T.hk[threadIdx.x] = 0;
  if (threadIdx.x == 0) {
    T.mean = s / P;
    T.sr = sr;
    T.pmn = pmn;
    T.pmx = pmx;
    T.ks = ks;
    T.kmn = kmn;
    T.kmx = kmx;
  }
}

// Contrast moments about the mean (Moments4, tamura.cpp:10-28) and the two
// histograms of one TAM_CHUNK of pixels.  By a block of 256.
__device__ __forceinline__ void tam_hist(const Img &im, const double *scr, int chunk, TamSum &T, TamPart2 *part) {
  __shared__ double shd[4];
  __shared__ int hk[3], hd[125];
  const long P = (long)im.h * im.w, c0 = (long)chunk * TAM_CHUNK;
  const gptr<const double> N = to_global(scr);
  const gptr<const double> phi = N + 2 * P;
  const gptr<const int> kb = (gptr<const int>)(N + 4 * P);
  const double mean = T.mean, pmn = T.pmn, kmn = T.kmn;
  const double ksc = hist_scale(kmn, (double)T.kmx, 3), psc = hist_scale(pmn, T.pmx, 125);
  if (threadIdx.x < 3) hk[threadIdx.x] = 0;
  if (threadIdx.x < 125) hd[threadIdx.x] = 0;
  __syncthreads();
  double m2 = 0, m4 = 0;
  int wk0 = 0, wk1 = 0, wk2 = 0;
  for (int r = 0; r < min((long)TAM_CHUNK, P - c0); r += 256 * 4) {
    double v[4], p[4];
    int kk[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const long i = min(c0 + r + 256 * k + threadIdx.x, P - 1);
      v[k] = N[i];
      p[k] = phi[i];
      kk[k] = kb[i];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const bool ok = c0 + r + 256 * k + threadIdx.x < P;
      int b = -1;
      if (ok) {
        const double d = v[k] - mean, d2 = d * d;
        m2 += d2;
        m4 += d2 * d2;
        b = hist_bin((double)kk[k], kmn, ksc, 3);
        atomicAdd(&hd[hist_bin(p[k], pmn, psc, 125)], 1);
      }
      wk0 += __popcll(__ballot(b == 0));
      wk1 += __popcll(__ballot(b == 1));
      wk2 += __popcll(__ballot(b == 2));
    }
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&hk[0], wk0);
    atomicAdd(&hk[1], wk1);
    atomicAdd(&hk[2], wk2);
  }
  __syncthreads();
  if (threadIdx.x < 3 && hk[threadIdx.x]) atomicAdd(&T.hk[threadIdx.x], hk[threadIdx.x]);
  if (threadIdx.x < 125 && hd[threadIdx.x]) atomicAdd(&T.hd[threadIdx.x], hd[threadIdx.x]);
  m2 = block_reduce(m2, SumOp(), shd);
  m4 = block_reduce(m4, SumOp(), shd);
  if (threadIdx.x == 0) part[chunk] = TamPart2{m2, m4};
}

// The features.  By a wave or more of a block.
__device__ __forceinline__ void tam_final(const Img &im, const TamSum &T, const TamPart2 *part, double *out) {
  __shared__ double shd[4];
  const int H = im.h, W = im.w;
  const long P = (long)H * W;
  double m2 = 0, m4 = 0;
  for (long b = threadIdx.x; b < (P + TAM_CHUNK - 1) / TAM_CHUNK; b += blockDim.x) {
    m2 += part[b].m2;
    m4 += part[b].m4;
  }
  m2 = block_reduce(m2, SumOp(), shd);
  m4 = block_reduce(m4, SumOp(), shd);
  if (threadIdx.x == 0) {
    const int *hk = T.hk, *hd = T.hd;
    const long long ks = T.ks;
    const double sr = T.sr;
    // coarseness (tamura.cpp:240-262); the divisor is unsigned arithmetic
    const unsigned xD = W, yD = H;
    double sum = (double)ks;
    if (yD == 32 || xD == 32) sum /= ((xD + 1 - 32) * (yD + 1 - 32));
    else sum /= ((yD - 32) * (xD - 32));
    double hm = 0;
    for (int k = 0; k < 3; k++) if (hk[k] > hm) hm = hk[k];
    // directionality (tamura.cpp:75-101)
    double mxh = 0.0;
    long fmx = 0;
    for (long a = 0; a < 125; a++) if (hd[a] > mxh) { mxh = hd[a]; fmx = a; }
    double ssum = 0;
    for (long a = 0; a < 125; a++) ssum += hd[a] * (double)((a + 1 - fmx) * (a + 1 - fmx));
    const double dir = fabs(log(ssum / sr + 0.0000001));
    // contrast
    double con;
    const double stdv = P > 2 ? sqrt(m2 / (P - 1)) : 0.0;
    const double kurt = P > 4 ? (P * m4) / (m2 * m2) : 0.0;
    if (stdv < kDblEps) con = 0;
    else con = stdv / pow(kurt / pow(stdv, 4), 0.25);
    out[0] = hk[0] / hm;
    out[1] = hk[1] / hm;
    out[2] = hk[2] / hm;
    out[3] = con;
    out[4] = dir;
    out[5] = sum;
  }
}

// Planes of more than one chunk take three launches.  The others, which would
// wait for launches more than work, take one, their sums in LDS: 2,000 planes of
// 16 x 16 46 us, 117 by three launches.
__device__ __forceinline__ TamSum &tam_sum(const Img &im, double *scr) { return *(TamSum *)(scr + tam_summary((long)im.h * im.w)); }
__device__ __forceinline__ TamPart2 *tam_part2(const Img &im, double *scr) { return (TamPart2 *)(scr + tam_parts2(im.h, im.w)); }
__global__ void __launch_bounds__(256) k_tam_mid(const Img *imgs, double *const *scr) {
  const Img im = imgs[blockIdx.x];
  if ((long)im.h * im.w > TAM_CHUNK) tam_mid(im, scr[blockIdx.x], tam_sum(im, scr[blockIdx.x]));
}
__global__ void __launch_bounds__(256) k_tam_hist(const Img *imgs, double *const *scr) {
  const Img im = imgs[blockIdx.y];
  const long P = (long)im.h * im.w;
  double *const q = scr[blockIdx.y];
  if (P > TAM_CHUNK && (long)blockIdx.x * TAM_CHUNK < P) tam_hist(im, q, blockIdx.x, tam_sum(im, q), tam_part2(im, q));
}
__global__ void __launch_bounds__(64) k_tam_final(const Img *imgs, double *const *scr, OutRef o) {
  const Img im = imgs[blockIdx.x];
  double *const q = scr[blockIdx.x];
  if ((long)im.h * im.w > TAM_CHUNK) tam_final(im, tam_sum(im, q), tam_part2(im, q), o.rows[blockIdx.x]);
}
__global__ void __launch_bounds__(256) k_tam_small(const Img *imgs, double *const *scr, OutRef o) {
  __shared__ TamSum sum;
  __shared__ TamPart2 part;
  const Img im = imgs[blockIdx.x];
  if ((long)im.h * im.w > TAM_CHUNK) return;
  tam_mid(im, scr[blockIdx.x], sum);
  __syncthreads();
  tam_hist(im, scr[blockIdx.x], 0, sum, &part);
  __syncthreads();
  tam_final(im, sum, &part, o.rows[blockIdx.x]);
}

void launch_tamura(const Img *imgs, const Stats *st, double *const *scratch, OutRef o, int nimg, int maxh, int maxw,
                   hipStream_t s) {
  const long maxn = (long)maxh * maxw;
  const int blocks = (tam_max_runs(maxh, maxw) + 3) / 4;
  const int nblocks = (int)((maxn / 4 + 255) / 256), sat = std::min((maxh + 63) / 64, SAT_WAVES);
  k_tam_norm<<<dim3(nblocks < 1 ? 1 : (nblocks > 1024 ? 1024 : nblocks), nimg), 256, 0, s>>>(imgs, st, scratch);
  static const bool lds_ok = hipFuncSetAttribute((const void *)k_tam_sat, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                  SAT_WAVES * (SAT_TILE + 64) * sizeof(double)) == hipSuccess;
  (void)lds_ok;
  k_tam_sat<<<nimg, 64 * sat, sat * (SAT_TILE + 64) * sizeof(double), s>>>(imgs, scratch);
  k_tam_pix<<<xcd_grid(blocks, nimg), 256, 0, s>>>(imgs, scratch, nimg, blocks);
  if (maxn > TAM_CHUNK) {
    k_tam_mid<<<nimg, 256, 0, s>>>(imgs, scratch);
    k_tam_hist<<<dim3((unsigned)((maxn + TAM_CHUNK - 1) / TAM_CHUNK), nimg), 256, 0, s>>>(imgs, scratch);
    k_tam_final<<<nimg, 64, 0, s>>>(imgs, scratch, o);
  }
  k_tam_small<<<nimg, 256, 0, s>>>(imgs, scratch, o);
}

// ================================================================= Comb moments
// CombFirst4Moments2D (CombFirst4Moments.cpp:78-217): 4 combs x 20 lines, one
// thread per line running the reference's sequential Moments4 over the
// line's pixels in raster order.  iis[img*20 + j] are the 20 rounded line
// offsets (host-computed with the reference's FP accumulation), NaN = unused.
__global__ void __launch_bounds__(128) k_comb(const Img *imgs, const double *iis, OutRef o) {
  __shared__ double mm[4][4][20];
  const Img im = imgs[blockIdx.x];
  const long m = im.h, n = im.w;
  const long n2 = n / 2, m2 = m / 2;
  const int t = threadIdx.x;
  if (t < 80) {
    const int comb = t / 20, li = t % 20;
    const double iid = iis[blockIdx.x * 20 + li];
    double z[4] = {0, 0, 0, 0};
    if (iid == iid) {
      const long ii = (long)iid;
      double mean = 0, M2 = 0, M3 = 0, M4 = 0;
      size_t cnt = 0;
      auto add = [&](double x) {
        if (!moments_ok(x)) return;
        const size_t n1 = cnt;
        cnt = cnt + 1;
        const double delta = x - mean;
        const double delta_n = delta / cnt;
        const double delta_n2 = delta_n * delta_n;
        const double term1 = delta * delta_n * n1;
        mean = mean + delta_n;
        M4 = M4 + term1 * delta_n2 * (cnt * cnt - 3 * cnt + 3) + 6 * delta_n2 * M2 - 4 * delta_n * M3;
        M3 = M3 + term1 * delta_n * (cnt - 2) - 3 * delta_n * M2;
        M2 = M2 + term1;
      };
      if (comb == 0) {         // |I + ii - J| < 1  ->  x = y + ii
        for (long y = 0; y < m; y++) { const long x = y + ii; if (x >= 0 && x < n) add(im.p[y * n + x]); }
      } else if (comb == 1) {  // J1 = n - x  ->  x = n - 1 - y - ii
        for (long y = 0; y < m; y++) { const long x = n - 1 - y - ii; if (x >= 0 && x < n) add(im.p[y * n + x]); }
      } else if (comb == 2) {  // vertical: x = n2 - 1 - ii
        const long x = n2 - 1 - ii;
        if (x >= 0 && x < n) for (long y = 0; y < m; y++) add(im.p[y * n + x]);
      } else {                 // horizontal: y = m2 - 1 - ii
        const long y = m2 - 1 - ii;
        if (y >= 0 && y < m) for (long x = 0; x < n; x++) add(im.p[y * n + x]);
      }
      z[0] = mean;
      z[1] = cnt > 2 ? sqrt(M2 / (cnt - 1)) : 0.0;
      z[2] = cnt > 3 ? (sqrt((double)cnt) * M3) / pow(M2, 1.5) : 0.0;
      z[3] = cnt > 4 ? (cnt * M4) / (M2 * M2) : 0.0;
    }
    for (int a = 0; a < 4; a++) mm[comb][a][li] = z[a];
  }
  __syncthreads();
  if (t == 0) {
    double vec[48];
    int vi = 0;
    for (int comb = 0; comb < 4; comb++)
      for (int a = 0; a < 4; a++) {
        double hmin = kInf, hmax = -kInf;
        for (int b = 0; b < 20; b++) { const double v = mm[comb][a][b]; if (v > hmax) hmax = v; if (v < hmin) hmin = v; }
        const double hs = hist_scale(hmin, hmax, 3);
        double bins[3] = {0, 0, 0};
        for (int b = 0; b < 20; b++) bins[hist_bin(mm[comb][a][b], hmin, hs, 3)] += 1.0;
        for (int b = 0; b < 3; b++) vec[vi++] = bins[b];
      }
    const int ord[48] = {45, 46, 47, 36, 37, 38, 42, 43, 44, 39, 40, 41, 33, 34, 35, 24,
                         25, 26, 30, 31, 32, 27, 28, 29, 9, 10, 11, 0, 1, 2, 6, 7,
                         8, 3, 4, 5, 21, 22, 23, 12, 13, 14, 18, 19, 20, 15, 16, 17};
    double *out = o.rows[blockIdx.x];
    for (int a = 0; a < 48; a++) out[a] = vec[ord[a]];
  }
}

void launch_comb(const Img *imgs, const double *iis, OutRef o, int nimg, hipStream_t s) {
  k_comb<<<nimg, 128, 0, s>>>(imgs, iis, o);
}

// ======================================================================== Radon
// radon.cpp:14-91 restated as a gather: each projection bin r of angle a sums,
// in the reference's (n, m) scan order, pixelLow of sub-pixels with
// floor(rIdx) == r and (pixel - pixelLow) of those with floor(rIdx) == r-1.
// floor(rIdx(n, m)) is non-increasing in m, so each column n contributes a
// contiguous m-range found by binary search.  trig[4][2] = {cos, sin} (glibc).
__device__ __forceinline__ double radon_ridx(int n, int m, int M, int N, double cs, double sn, int rFirst) {
  const int xO = (N - 1) / 2, yO = (M - 1) / 2;
  const double xT = (-xO - 0.25) + 0.5 * n;
  const double yT = (-yO - 0.25) + 0.5 * (2 * M - 1 - m);
  const double xc = xT * cs - rFirst;
  const double ys = yT * sn;
  return xc + ys;
}

// Block = (angle, group of 256 bins, image); thread = bin r.  The y*sin
// table of the reference (radon.cpp:58-63) is built in LDS and x*cos
// recomputed with the reference's operations, so rIdx is bit-identical.
// floor(rIdx) is monotone in the sub-column n (x*cos is) and non-increasing
// in the sub-row m, so the sub-columns touching bin r form an interval
// (binary search) and, per sub-column, the sub-rows with floor(rIdx) in
// {r-1, r} form a range that moves slowly with n (tracked by stepping).
// Each bin's terms are added in the reference's order: sub-columns
// ascending, sub-rows ascending within one.
//   At angle 0 a bin is a pixel column and the lanes of a wave read
// adjacent pixels of one row, so pixels are read from global memory
// directly.  At the other angles a lane follows its own slanted line, so a
// direct read touches one cache line per lane; there the block streams the
// plane through LDS in chunks of whole pixel columns (rows limited to the
// band its bins can reach, with a direct read as the fallback outside it),
// and every lane takes its sub-columns of a chunk in order.
// doubles of the LDS chunk buffer: 16 KB keeps 8 blocks per CU; the
// kernel is bound by each bin's sequential sum, and larger chunks (lower
// occupancy) measured slower
constexpr int RADON_TILE = 2048;
__device__ __forceinline__ double radon_xc(int nn, int xO, double cs, int rFirst) {
  return ((-xO - 0.25) + 0.5 * nn) * cs - rFirst;
}

__global__ void __launch_bounds__(256) k_radon_proj(const Img *imgs, const double *trig, double *const *proj,
                                                    int nbg, int nimg, int ysz, int a0, int na) {
  extern __shared__ double lds[];
  double *yS = lds, *tile = lds + ysz;
  __shared__ int ired[8];
  int ent, sub;
  if (!xcd_item(na * nbg, nimg, ent, sub)) return;
  const Img im = imgs[ent];
  const int M = im.h, N = im.w;
  const int rLast = (int)ceil(sqrt((double)((N - 1 - (N - 1) / 2) * (N - 1 - (N - 1) / 2)) +
                                   (double)((M - 1 - (M - 1) / 2) * (M - 1 - (M - 1) / 2)))) + 1;
  const int rFirst = -rLast, rSize = rLast - rFirst + 1;
  const int a = a0 + sub / nbg, r0 = (sub % nbg) * 256;
  if (r0 >= rSize) return;
  const double cs = trig[2 * a], sn = trig[2 * a + 1];
  const int xO = (N - 1) / 2, yO = (M - 1) / 2;
  const int M2 = 2 * M, N2 = 2 * N;
  for (int p = threadIdx.x; p < M2; p += blockDim.x) yS[p] = ((-yO - 0.25) + 0.5 * (M2 - 1 - p)) * sn;
  __syncthreads();
  const int r = r0 + threadIdx.x;
  const bool act = r < rSize;
  const double yS0 = yS[0], ySL = yS[M2 - 1];
  // column nn is skipped when floor(xc + yS0) < r-1 (A) or floor(xc + ySL) > r (B)
  auto predA = [&](int nn) { return (int)(radon_xc(nn, xO, cs, rFirst) + yS0) < r - 1; };
  auto predB = [&](int nn) { return (int)(radon_xc(nn, xO, cs, rFirst) + ySL) > r; };
  int lo = 0, hi = N2;
  if (!act) {
    hi = 0;
  } else if (cs > 0) {  // A: true then false; B: false then true
    int l = 0, h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (!predA(mid)) h = mid; else l = mid + 1; }
    lo = l;
    l = lo; h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (predB(mid)) h = mid; else l = mid + 1; }
    hi = l;
  } else if (cs < 0) {  // B: true then false; A: false then true
    int l = 0, h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (!predB(mid)) h = mid; else l = mid + 1; }
    lo = l;
    l = lo; h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (predA(mid)) h = mid; else l = mid + 1; }
    hi = l;
  } else if (predA(0) || predB(0)) {
    hi = 0;
  }
  const gptr<const double> P = to_global((const double *)im.p);
  double acc = 0.0;
  int m0 = 0, m1 = 0;
  // sub-rows [m0, m1) of column nn whose bin is r or r-1; [m0, m1) moves
  // monotonically with nn
  auto range = [&](int nn, double xc) {
    if (nn == lo) {
      int l = 0, h = M2;
      while (l < h) { const int mid = (l + h) >> 1; if ((int)(xc + yS[mid]) <= r) h = mid; else l = mid + 1; }
      m0 = l;
      l = m0; h = M2;
      while (l < h) { const int mid = (l + h) >> 1; if ((int)(xc + yS[mid]) < r - 1) h = mid; else l = mid + 1; }
      m1 = l;
    } else {
      while (m0 > 0 && (int)(xc + yS[m0 - 1]) <= r) m0--;
      while (m0 < M2 && (int)(xc + yS[m0]) > r) m0++;
      if (m1 < m0) m1 = m0;
      while (m1 > m0 && (int)(xc + yS[m1 - 1]) < r - 1) m1--;
      while (m1 < M2 && (int)(xc + yS[m1]) >= r - 1) m1++;
    }
  };
  auto term = [&](double pixel, double xc, int mm) {
    if (pixel) {
      pixel *= 0.25;
      const double rIdx = (xc + yS[mm]);
      const int rLow = (int)rIdx;
      const double pixelLow = pixel * (1 - rIdx + rLow);
      if (rLow == r) acc += pixelLow;
      else acc += pixel - pixelLow;
    }
  };
  if (fabs(sn) < 0.5) {  // angle 0: lanes read adjacent pixels of a row
    for (int nn = lo; nn < hi; nn++) {
      const double xc = radon_xc(nn, xO, cs, rFirst);
      range(nn, xc);
      const gptr<const double> col = P + (nn >> 1);
#pragma unroll 4
      for (int mm = m0; mm < m1; mm++) term(col[(unsigned)((mm >> 1) * N)], xc, mm);
    }
    if (act) proj[ent][(long)a * rSize + r] = acc;
    return;
  }
  // pixel columns any bin of the block touches
  const int xlo = block_reduce(lo < hi ? lo >> 1 : N, MinOp(), ired);
  const int xhi = block_reduce(lo < hi ? (hi + 1) >> 1 : 0, MaxOp(), ired);
  const int Wc = max(1, min(32, RADON_TILE / (M + 1)));  // wc * ld <= RADON_TILE (ld <= M + 1)
  const int r1 = min(r0 + 256, rSize);
  int nn = lo;
  for (int x0 = xlo; x0 < xhi; x0 += Wc) {
    const int x1 = min(x0 + Wc, N), wc = x1 - x0;
    // rows the block's bins [r0, r1) can reach in sub-columns [2 x0, 2 x1):
    // floor(rIdx) in [r0 - 1, r1 - 1] with rIdx = xc + yS(mm) and
    // yS(mm) = (-yO - 0.25 + 0.5 (M2 - 1 - mm)) sn, sn > 0; two rows of margin
    const double xa = radon_xc(2 * x0, xO, cs, rFirst), xb = radon_xc(2 * x1 - 1, xO, cs, rFirst);
    const double xcmin = fmin(xa, xb), xcmax = fmax(xa, xb);
    const double c0 = -yO - 0.25;
    const double mlo = (M2 - 1) - 2 * ((r1 - xcmin) / sn - c0);
    const double mhi = (M2 - 1) - 2 * ((r0 - 1 - xcmax) / sn - c0);
    const int rb0 = max(0, (int)floor(fmax(mlo, -4.0) * 0.5) - 2);
    const int rb1 = min(M, (int)floor(fmin(mhi, (double)M2 + 4) * 0.5) + 3);
    const int band = max(0, rb1 - rb0);
    const int ld = band | 1;  // odd stride: column reads of adjacent rows fall in different banks
    __syncthreads();  // the previous chunk is consumed
    for (int e = threadIdx.x; e < wc * band; e += blockDim.x) {
      const int row = e / wc, c = e - row * wc;
      tile[c * ld + row] = P[(long)(rb0 + row) * N + x0 + c];
    }
    __syncthreads();
    const int nend = min(hi, 2 * x1);
    for (; nn < nend; nn++) {
      const double xc = radon_xc(nn, xO, cs, rFirst);
      range(nn, xc);
      const int c = (nn >> 1) - x0;
      for (int mm = m0; mm < m1; mm++) {
        const int row = mm >> 1;
        const double pixel = (row >= rb0 && row < rb1) ? tile[c * ld + row - rb0] : P[(long)row * N + (nn >> 1)];
        term(pixel, xc, mm);
      }
    }
  }
  if (act) proj[ent][(long)a * rSize + r] = acc;
}

// yTable / xTable entries are exact multiples of 0.25, so the closed forms
// above equal the reference's running sums.
__global__ void k_radon_hist(const Img *imgs, double *const *proj, OutRef o) {
  const Img im = imgs[blockIdx.x];
  const int M = im.h, N = im.w;
  const int rLast = (int)ceil(sqrt((double)((N - 1 - (N - 1) / 2) * (N - 1 - (N - 1) / 2)) +
                                   (double)((M - 1 - (M - 1) / 2) * (M - 1 - (M - 1) / 2)))) + 1;
  const int rSize = 2 * rLast + 1;
  if (threadIdx.x != 0) return;
  double v[12];
  int vi = 0;
  for (int a = 0; a < 4; a++) {
    const double *p = proj[blockIdx.x] + (long)a * rSize;
    double hmin = kInf, hmax = -kInf;
    for (int i = 0; i < rSize; i++) { if (p[i] > hmax) hmax = p[i]; if (p[i] < hmin) hmin = p[i]; }
    const double hs = hist_scale(hmin, hmax, 3);
    double bins[3] = {0, 0, 0};
    for (int i = 0; i < rSize; i++) bins[hist_bin(p[i], hmin, hs, 3)] += 1.0;
    for (int b = 0; b < 3; b++) v[vi++] = bins[b];
  }
  const int ord[12] = {0, 1, 2, 9, 10, 11, 3, 4, 5, 6, 7, 8};
  double *out = o.rows[blockIdx.x];
  for (int a = 0; a < 12; a++) out[a] = v[ord[a]];
}

// --------------------------------------------------- certified (order-free) form
// A projection bin of the reference is the sequential sum of its terms.  Any
// other summation of the same terms lies within gamma_K * sum|terms| of their
// exact sum, as does the reference's (K bounds the depth of both summation
// trees), so the reference's bin lies within 2 gamma_K sum|terms| of an
// order-free sum.  The 12 features only need each bin's 3-bin histogram slot
// and the extreme bins of each angle: k_radon_sum forms the order-free sums
// with a bound per bin, and k_radon_cert settles the extremes and every slot
// from them, recomputing in the reference's order the bins a bound leaves
// open.  The counts equal the reference's bit for bit.

// LDS of one wave's recomputation: the terms of one window, and per
// sub-column of a chunk the offset of its first term and its first sub-row
constexpr int RADON_RTB = 512;  // terms per window (8 per lane)
constexpr int RADON_RCH = 256;  // sub-columns per chunk (4 per lane)
struct RadonWaveLds {
  double tb[RADON_RTB];
  int off[RADON_RCH];
  int m0[RADON_RCH];
};

// Bin r of the projection at (cs, sn) in the reference's order (radon.cpp:
// 66-81: sub-columns ascending, sub-rows ascending within one), by the 64
// lanes of a wave (r uniform).  Per chunk of 256 sub-columns each lane finds
// the sub-rows of four (those whose floor(rIdx) is r or r-1, a range, as
// floor(rIdx) is non-increasing in the sub-row), a wave scan turns the counts
// into offsets, the lanes form the terms 512 at a time into LDS in the
// reference's order with its operations (8 pixel loads in flight per lane),
// and lane 0 adds them in that order.  A zero pixel, which the reference
// skips, gives a +0 term (the running sum is never -0, so adding +0 leaves it
// unchanged).  Every lane returns the sum.
__device__ double radon_bin_wave(gptr<const double> P, int M, int N, double cs, double sn, int rFirst, int r,
                                 RadonWaveLds &W) {
  const int lane = threadIdx.x & 63;
  const int xO = (N - 1) / 2, yO = (M - 1) / 2, M2 = 2 * M, N2 = 2 * N;
  auto yS = [&](int mm) { return ((-yO - 0.25) + 0.5 * (M2 - 1 - mm)) * sn; };
  const double yS0 = yS(0), ySL = yS(M2 - 1);
  auto predA = [&](int nn) { return (int)(radon_xc(nn, xO, cs, rFirst) + yS0) < r - 1; };
  auto predB = [&](int nn) { return (int)(radon_xc(nn, xO, cs, rFirst) + ySL) > r; };
  int lo = 0, hi = N2;
  if (cs > 0) {
    int l = 0, h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (!predA(mid)) h = mid; else l = mid + 1; }
    lo = l;
    l = lo; h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (predB(mid)) h = mid; else l = mid + 1; }
    hi = l;
  } else if (cs < 0) {
    int l = 0, h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (!predB(mid)) h = mid; else l = mid + 1; }
    lo = l;
    l = lo; h = N2;
    while (l < h) { const int mid = (l + h) >> 1; if (predA(mid)) h = mid; else l = mid + 1; }
    hi = l;
  } else if (predA(0) || predB(0)) {
    hi = 0;
  }
  double acc = 0.0;
  for (int cb = lo; cb < hi; cb += RADON_RCH) {
    int cnt[4], mlo[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int nn = cb + 4 * lane + k;
      int m0 = 0, m1 = 0;
      if (nn < hi) {
        const double xc = radon_xc(nn, xO, cs, rFirst);
        int l = 0, h = M2;
        while (l < h) { const int mid = (l + h) >> 1; if ((int)(xc + yS(mid)) <= r) h = mid; else l = mid + 1; }
        m0 = l;
        h = M2;
        while (l < h) { const int mid = (l + h) >> 1; if ((int)(xc + yS(mid)) < r - 1) h = mid; else l = mid + 1; }
        m1 = l;
      }
      cnt[k] = m1 - m0;
      mlo[k] = m0;
    }
    const int own = cnt[0] + cnt[1] + cnt[2] + cnt[3];
    int inc = own;
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    const int total = __shfl(inc, 63, 64);
    int ofs = inc - own;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      W.off[4 * lane + k] = ofs;
      W.m0[4 * lane + k] = mlo[k];
      ofs += cnt[k];
    }
    wave_sync();
    for (int w0 = 0; w0 < total; w0 += RADON_RTB) {
      const int wn = min(RADON_RTB, total - w0);
      int nj[8], mj[8];
      double px[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int g = w0 + min(lane + 64 * i, wn - 1);
        int j = 0;  // the sub-column holding term g: the last j with off[j] <= g
        for (int st = RADON_RCH / 2; st > 0; st >>= 1)
          if (W.off[j + st] <= g) j += st;
        nj[i] = cb + j;
        mj[i] = W.m0[j] + (g - W.off[j]);
        px[i] = P[(long)(mj[i] >> 1) * N + (nj[i] >> 1)];
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int t = lane + 64 * i;
        if (t < wn) {
          double pixel = px[i], term = 0.0;
          if (pixel) {
            pixel *= 0.25;
            const double rIdx = (radon_xc(nj[i], xO, cs, rFirst) + yS(mj[i]));
            const int rLow = (int)rIdx;
            const double pixelLow = pixel * (1 - rIdx + rLow);
            term = (rLow == r) ? pixelLow : pixel - pixelLow;
          }
          W.tb[t] = term;
        }
      }
      wave_sync();
      if (lane == 0) {
        int i = 0;
        for (; i + 8 <= wn; i += 8) {
          double t8[8];
#pragma unroll
          for (int k = 0; k < 8; k++) t8[k] = W.tb[i + k];
#pragma unroll
          for (int k = 0; k < 8; k++) acc += t8[k];
        }
        for (; i < wn; i++) acc += W.tb[i];
      }
      wave_sync();  // the window is consumed
    }
  }
  return __shfl(acc, 0, 64);
}

template <typename T, typename Op>
__device__ __forceinline__ T wave_all_reduce(T v, Op op) {
  for (int o = 32; o > 0; o >>= 1) v = op(v, __shfl_xor(v, o, 64));
  return v;
}

// Order-free projection sums.  Block = (group of NA angles, image plane); a
// thread walks pixel columns top to bottom (the lanes of a wave read adjacent
// pixels of a row).  Each sub-pixel's two terms are the reference's
// (radon.cpp:66-81: the same rIdx, rLow, pixelLow and pixel - pixelLow).  Down
// a column rIdx is non-increasing, and the four sub-pixels of a pixel span
// less than one unit of it, so a pixel's terms fall in bins pb..pb+2 (pb =
// its smallest rLow) and pb never rises: the thread keeps the sums of those
// three bins in registers and adds a bin into the block's LDS copy of the
// projection (a double atomic) once the column has left it.  The terms go
// into the window with fused multiply-adds by 0 or 1, exact products, so
// each term is added by one rounding.  Beside each sum, W accumulates |pixel|
// over every pixel whose window holds the bin: each term is at most
// |pixel| / 4 (1 + 2^-39), so W bounds the bin's sum|terms|.
// Output per plane: sums at [a][r], bounds at [4 + a][r].
template <int NA>
__global__ void __launch_bounds__(256) k_radon_sum(const Img *imgs, const double *trig, double *const *proj, int ngrp,
                                                   int nimg) {
  extern __shared__ double lds[];
  int ent, grp;
  if (!xcd_item(ngrp, nimg, ent, grp)) return;
  const Img im = imgs[ent];
  const int M = im.h, N = im.w;
  const int rLast = (int)ceil(sqrt((double)((N - 1 - (N - 1) / 2) * (N - 1 - (N - 1) / 2)) +
                                   (double)((M - 1 - (M - 1) / 2) * (M - 1 - (M - 1) / 2)))) + 1;
  const int rFirst = -rLast, rSize = 2 * rLast + 1;
  const int a0 = grp * NA;
  double *S = lds, *W = lds + NA * rSize;
  for (int i = threadIdx.x; i < 2 * NA * rSize; i += blockDim.x) lds[i] = 0.0;
  __syncthreads();
  const int xO = (N - 1) / 2, yO = (M - 1) / 2, M2 = 2 * M;
  double cs[NA], sn[NA];
#pragma unroll
  for (int a = 0; a < NA; a++) {
    cs[a] = trig[2 * (a0 + a)];
    sn[a] = trig[2 * (a0 + a) + 1];
  }
  const gptr<const double> P = to_global((const double *)im.p);
  const double c0 = -yO - 0.25;
  // a bin's sum into LDS; w == 0 means no nonzero pixel reached it (s == +0)
  auto flush = [&](int a, int b, double sv, double wv) {
    if (wv != 0.0) {
      b = min(max(b, 0), rSize - 1);
      atomicAdd(&S[a * rSize + b], sv);
      atomicAdd(&W[a * rSize + b], wv);
    }
  };
  for (int c = threadIdx.x; c < N; c += blockDim.x) {
    double xa[NA], xb[NA], R0[NA], R1[NA], R2[NA], A0[NA], A1[NA], A2[NA];
    double base[NA];  // the window's first bin
#pragma unroll
    for (int a = 0; a < NA; a++) {
      xa[a] = radon_xc(2 * c, xO, cs[a], rFirst);
      xb[a] = radon_xc(2 * c + 1, xO, cs[a], rFirst);
      R0[a] = R1[a] = R2[a] = A0[a] = A1[a] = A2[a] = 0.0;
      base[a] = 1e9;  // above every bin: the first pixel opens the window
    }
    double pn = P[c];
    for (int y = 0; y < M; y++) {
      const double pix = pn;
      if (y + 1 < M) pn = P[(long)(y + 1) * N + c];
      const double q = pix * 0.25, ap = fabs(pix);
      // yTable of sub-rows 2y and 2y+1 (exact multiples of 0.25)
      const double ya = c0 + 0.5 * (M2 - 1 - 2 * y), yb = ya - 0.5;
#pragma unroll
      for (int a = 0; a < NA; a++) {
        const double ysa = ya * sn[a], ysb = yb * sn[a];
        const double r00 = xa[a] + ysa, r01 = xa[a] + ysb, r10 = xb[a] + ysa, r11 = xb[a] + ysb;
        // rLow = (int)rIdx as a double (rIdx >= 0 is far below 2^31)
        const double l00 = trunc(r00), l01 = trunc(r01), l10 = trunc(r10), l11 = trunc(r11);
        const double pb = fmin(fmin(l00, l01), fmin(l10, l11));
        if (pb < base[a]) {
          if (base[a] - pb >= 3.0) {
            flush(a, (int)base[a], R0[a], A0[a]);
            flush(a, (int)base[a] + 1, R1[a], A1[a]);
            flush(a, (int)base[a] + 2, R2[a], A2[a]);
            R0[a] = R1[a] = R2[a] = A0[a] = A1[a] = A2[a] = 0.0;
          } else {
            do {
              flush(a, (int)base[a] + 2, R2[a], A2[a]);
              R2[a] = R1[a]; R1[a] = R0[a]; R0[a] = 0.0;
              A2[a] = A1[a]; A1[a] = A0[a]; A0[a] = 0.0;
              base[a] -= 1.0;
            } while (pb < base[a]);
          }
          base[a] = pb;
        }
        auto add = [&](double rIdx, double rLow) {
          const double pixelLow = q * (1 - rIdx + rLow), pixelHigh = q - pixelLow;
          const double d = rLow - pb, e = 1.0 - d;  // rLow - pb is 0 or 1
          R0[a] = fma(e, pixelLow, R0[a]);
          R1[a] = fma(d, pixelLow, R1[a]);
          R1[a] = fma(e, pixelHigh, R1[a]);
          R2[a] = fma(d, pixelHigh, R2[a]);
        };
        add(r00, l00);
        add(r01, l01);
        add(r10, l10);
        add(r11, l11);
        A0[a] += ap;
        A1[a] += ap;
        A2[a] += ap;
      }
    }
#pragma unroll
    for (int a = 0; a < NA; a++) {
      flush(a, (int)base[a], R0[a], A0[a]);
      flush(a, (int)base[a] + 1, R1[a], A1[a]);
      flush(a, (int)base[a] + 2, R2[a], A2[a]);
    }
  }
  __syncthreads();
  double *out = proj[ent];
  for (int i = threadIdx.x; i < NA * rSize; i += blockDim.x) {
    out[(long)a0 * rSize + i] = S[i];
    out[(long)(4 + a0) * rSize + i] = W[i];
  }
}

// Per plane (block of 256): wave a takes angle a.  The bins whose interval
// [sum - d, sum + d], d = 4 gamma_K W slack, reaches the smallest upper end
// or the largest lower end are the only ones that can be the minimum or the
// maximum; they are recomputed in the reference's order, which gives the
// reference's hmin and hmax exactly.  A bin's slot is then decided from its
// interval (hist_bin is monotone in the value) or, when the interval straddles
// a slot boundary, from its recomputed value.  K = 4MN + 4M + N + 8 bounds the
// number of additions on any path of either summation tree.  Non-finite sums
// take the reference's path for that angle: every bin recomputed, the
// histogram formed serially as radon.cpp does.
__global__ void __launch_bounds__(256) k_radon_cert(const Img *imgs, const double *trig, double *const *proj,
                                                    OutRef o, double slack) {
  __shared__ RadonWaveLds wl[4];
  __shared__ double v[12];  // the 12 counts, angle-major
  const int a = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const Img im = imgs[blockIdx.x];
  const int M = im.h, N = im.w;
  const int rLast = (int)ceil(sqrt((double)((N - 1 - (N - 1) / 2) * (N - 1 - (N - 1) / 2)) +
                                   (double)((M - 1 - (M - 1) / 2) * (M - 1 - (M - 1) / 2)))) + 1;
  const int rFirst = -rLast, rSize = 2 * rLast + 1;
  const double K = 4.0 * M * N + 4.0 * M + N + 8.0, u = 0x1p-53;
  const double cb = 4.0 * (K * u / (1.0 - K * u)) * slack;
  // sums of subnormal-sized terms: a floor keeps d from underflowing to 0
  auto dlt = [&](double wv) { return wv > 0.0 ? fmax(cb * wv, 0x1p-1000) : 0.0; };
  const gptr<const double> P = to_global((const double *)im.p);
  double *const p = proj[blockIdx.x] + (long)a * rSize, *const w = proj[blockIdx.x] + (long)(4 + a) * rSize;
  const double cs = trig[2 * a], sn = trig[2 * a + 1];
  double L = __builtin_inf(), U = -__builtin_inf();
  bool nonfinite = false;
  for (int r = lane; r < rSize; r += 64) {
    const double d = dlt(w[r]), lo = p[r] - d, hi = p[r] + d;
    if (!(fabs(lo) <= 1.7976931348623157e308 && fabs(hi) <= 1.7976931348623157e308)) nonfinite = true;
    L = fmin(L, hi);
    U = fmax(U, lo);
  }
  L = wave_all_reduce(L, MinOp());
  U = wave_all_reduce(U, MaxOp());
  const bool bad = __ballot(nonfinite) != 0;
  // candidates (every bin when bad), each recomputed by the whole wave
  for (int c0 = 0; c0 < rSize; c0 += 64) {
    const int r = c0 + lane;
    bool need = false;
    if (r < rSize) {
      const double wv = w[r];
      if (bad ? wv != 0.0 : wv > 0.0) {
        const double d = dlt(wv), lo = p[r] - d, hi = p[r] + d;
        need = bad || lo <= L || hi >= U;
      }
    }
    for (unsigned long long m = __ballot(need); m; m &= m - 1) {
      const int k = __ffsll((long long)m) - 1;
      const double e = radon_bin_wave(P, M, N, cs, sn, rFirst, c0 + k, wl[a]);
      if (lane == k) {
        p[r] = e;
        w[r] = 0.0;
      }
    }
  }
  wave_sync();
  if (bad) {  // every bin is the reference's: its serial histogram
    if (lane == 0) {
      double hmin = kInf, hmax = -kInf;
      for (int i = 0; i < rSize; i++) { if (p[i] > hmax) hmax = p[i]; if (p[i] < hmin) hmin = p[i]; }
      const double hs = hist_scale(hmin, hmax, 3);
      double b0 = 0, b1 = 0, b2 = 0;
      for (int i = 0; i < rSize; i++) {
        const int b = hist_bin(p[i], hmin, hs, 3);
        b0 += b == 0 ? 1.0 : 0.0;
        b1 += b == 1 ? 1.0 : 0.0;
        b2 += b == 2 ? 1.0 : 0.0;
      }
      v[3 * a] = b0;
      v[3 * a + 1] = b1;
      v[3 * a + 2] = b2;
    }
  } else {
    // the minimum and maximum bins are among the recomputed (or exact) ones
    double mn = __builtin_inf(), mx = -__builtin_inf();
    for (int r = lane; r < rSize; r += 64) {
      if (w[r] == 0.0) {
        mn = fmin(mn, p[r]);
        mx = fmax(mx, p[r]);
      }
    }
    mn = wave_all_reduce(mn, MinOp());
    mx = wave_all_reduce(mx, MaxOp());
    const double hs = hist_scale(mn, mx, 3);
    int n0 = 0, n1 = 0, n2 = 0;
    for (int c0 = 0; c0 < rSize; c0 += 64) {
      const int r = c0 + lane;
      int b = -1;
      bool open = false;
      if (r < rSize) {
        const double wv = w[r], pv = p[r];
        if (wv == 0.0) {
          b = hist_bin(pv, mn, hs, 3);
        } else {
          const double d = dlt(wv);
          b = hist_bin(fmax(pv - d, mn), mn, hs, 3);
          open = hist_bin(fmin(pv + d, mx), mn, hs, 3) != b;
        }
      }
      for (unsigned long long m = __ballot(open); m; m &= m - 1) {
        const int k = __ffsll((long long)m) - 1;
        const double e = radon_bin_wave(P, M, N, cs, sn, rFirst, c0 + k, wl[a]);
        if (lane == k) b = hist_bin(e, mn, hs, 3);
      }
      n0 += b == 0;
      n1 += b == 1;
      n2 += b == 2;
    }
    n0 = wave_all_reduce(n0, SumOp());
    n1 = wave_all_reduce(n1, SumOp());
    n2 = wave_all_reduce(n2, SumOp());
    if (lane == 0) {
      v[3 * a] = n0;
      v[3 * a + 1] = n1;
      v[3 * a + 2] = n2;
    }
  }
  __syncthreads();
  // output order of vd_RadonTextures (radon.cpp:98-115): angles 0, 135, 45, 90
  if (threadIdx.x < 12) {
    const int t = threadIdx.x, src = t < 3 ? t : t < 6 ? t + 6 : t - 3;
    o.rows[blockIdx.x][t] = v[src];
  }
}

// rSize above which the certified form's LDS (16 bytes per bin and angle)
// does not fit one angle per block
constexpr int RADON_CERT_MAXBINS = 10240;

bool radon_certified_fits(int maxbins) { return maxbins <= RADON_CERT_MAXBINS; }

void launch_radon_certified(const Img *imgs, const double *trig, double *const *proj, OutRef o, int nimg, int maxbins,
                            double slack, hipStream_t s) {
  // angles per block: as many as keep the block's LDS near 48 KB
  const int na = (64 * maxbins <= 49152) ? 4 : (32 * maxbins <= 49152) ? 2 : 1;
  const size_t lds = (size_t)2 * na * maxbins * sizeof(double);
  static const bool lds_ok =
      hipFuncSetAttribute((const void *)k_radon_sum<1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          2 * RADON_CERT_MAXBINS * (int)sizeof(double)) == hipSuccess;
  (void)lds_ok;
  const int ngrp = 4 / na;
  if (na == 4)
    k_radon_sum<4><<<xcd_grid(ngrp, nimg), 256, lds, s>>>(imgs, trig, proj, ngrp, nimg);
  else if (na == 2)
    k_radon_sum<2><<<xcd_grid(ngrp, nimg), 256, lds, s>>>(imgs, trig, proj, ngrp, nimg);
  else
    k_radon_sum<1><<<xcd_grid(ngrp, nimg), 256, lds, s>>>(imgs, trig, proj, ngrp, nimg);
  k_radon_cert<<<nimg, 256, 0, s>>>(imgs, trig, proj, o, slack);
}

void launch_radon(const Img *imgs, const double *trig, double *const *proj, OutRef o, int nimg, int maxbins,
                  int maxh, int maxw, hipStream_t s) {
  (void)maxw;
  // LDS: the y*sin table (2 maxh <= 8192 doubles), then, for the slanted
  // angles, the chunk buffer
  static const bool lds_ok = hipFuncSetAttribute((const void *)k_radon_proj, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                  (2 * 4096 + RADON_TILE) * (int)sizeof(double)) == hipSuccess;
  (void)lds_ok;
  const int ysz = 2 * maxh;
  const int nbg = (maxbins + 255) / 256;
  // angle 0 (direct reads, small LDS for occupancy), then angles 1..3
  k_radon_proj<<<xcd_grid(nbg, nimg), 256, (size_t)ysz * sizeof(double), s>>>(imgs, trig, proj, nbg, nimg, ysz, 0, 1);
  k_radon_proj<<<xcd_grid(3 * nbg, nimg), 256, ((size_t)ysz + RADON_TILE) * sizeof(double), s>>>(imgs, trig, proj, nbg,
                                                                                                 nimg, ysz, 1, 3);
  k_radon_hist<<<nimg, 64, 0, s>>>(imgs, proj, o);
}

}  // namespace wnd
