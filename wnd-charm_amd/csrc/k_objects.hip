// Otsu / Inverse-Otsu object features, Prewitt edge features and Gabor
// textures.  FP64.  Integer outputs (thresholds, labels, areas, counts,
// Euler number) are exact; the connected components are canonicalised to
// the reference's raster-order labelling.
#include "common.hpp"
#include "kernels.hpp"
#include "blocksort.hpp"

namespace wnd {

// Otsu threshold of a plane (ImageMatrix::Otsu(dynamic), cmatrix.cpp:1520-1570):
// 1024-bin histogram over [mn, mx], then the reference's omega / myu / sigma
// recurrence.  The threshold of a filled 1024-bin histogram, by the whole
// block (every thread calls it; uniform result): the bin fractions
// hist[i] / wh and, once thread 0 has run the sequential prefix sums om / my
// (and myu[L-1]) with the reference's operations, each bin's between-class
// variance are formed in parallel; the threshold is the first bin of the
// largest variance above 0 (the reference's strict comparison from 0).
__device__ double otsu_threshold(const int *hist, long n, double mn, double mx) {
  __shared__ double pf[1024], om_s[1024], my_s[1024];
  __shared__ double red_d[32];
  __shared__ long long red_l[32];
  __shared__ double my_last_s;
  const double wh = (double)(unsigned)n;
  for (int i = threadIdx.x; i < 1024; i += blockDim.x) pf[i] = hist[i] / wh;
  __syncthreads();
  if (threadIdx.x == 0) {
    double om = pf[0], my = 0.0;
    for (int i = 0; i < 1023; i++) {
      if (i > 0) {
        om = om + pf[i];
        my = my + i * pf[i];
      }
      om_s[i] = om;
      my_s[i] = my;
    }
    my_last_s = my + 1023 * pf[1023];  // myu[L-1], by the operations of the recurrence
  }
  __syncthreads();
  const double my_last = my_last_s;
  double best = 0.0;
  long long bi = 1023;  // no variance above 0: threshold bin 0 (below)
  for (int i = threadIdx.x; i < 1023; i += blockDim.x) {
    const double om = om_s[i], my = my_s[i];
    double sg;
    if (om != 0.0 && om != 1.0) {
      const double d = my_last * om - my;
      sg = (d * d) / (om * (1.0 - om));
    } else sg = 0.0;
    if (sg > best) { best = sg; bi = i; }  // this thread's bins ascend: its first maximum
  }
  const double top = block_reduce(best, MaxOp(), red_d);
  long long cand = (top > 0.0 && best == top) ? bi : 1023;
  cand = block_reduce(cand, MinOp(), red_l);
  const int thr = top > 0.0 ? (int)cand : 0;
  return ((((double)thr / (double)(1023)) * (mx - mn)) + mn);
}

template <typename ValF>
__device__ double block_otsu(long n, double mn, double mx, ValF val, int *hist) {
  for (int b = threadIdx.x; b < 1024; b += blockDim.x) hist[b] = 0;
  __syncthreads();
  const double sc = hist_scale(mn, mx, 1024);
#pragma unroll 4
  for (long i = threadIdx.x; i < n; i += blockDim.x) atomicAdd(&hist[hist_bin(val(i), mn, sc, 1024)], 1);
  __syncthreads();
  return otsu_threshold(hist, n, mn, mx);
}

// ------------------------------------------------------------- union-find
// Labels point to smaller indices of their component, roots to themselves.
// find(lab, x) reads the chain, join(lab, a, b) links two components at the
// smaller root: in LDS within a strip of rows, by device-scope atomics between
// strips (blocks of other XCDs take part).
__device__ __forceinline__ int uf_find(volatile int *lab, int x) {
  while (true) {
    const int p = lab[x];
    if (p == x) return x;
    x = p;
  }
}
__device__ __forceinline__ int uf_find_device(int *lab, int x) {
  while (true) {
    const int p = __hip_atomic_load(&lab[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (p == x) return x;
    x = p;
  }
}
template <class Find>
__device__ __forceinline__ void uf_union(int *lab, int a, int b, Find find) {
  while (true) {
    a = find(a);
    b = find(b);
    if (a == b) return;
    if (a < b) { const int t = a; a = b; b = t; }
    const int old = atomicMin(&lab[a], b);
    if (old == a) return;
    a = old;
  }
}

// Object features (ImageMatrix::FeatureStatistics, cmatrix.cpp:1642-1717;
// bwlabel / GlobalCentroid / FeatureCentroid / EulerNumber,
// FeatureStatistics.cpp:44-254; output layout FeatureAlgorithms.cpp:370-394).
// invert != 0 evaluates the Inverse-Otsu variant on v' = (max - v) + min
// (ImageMatrix::invert, cmatrix.cpp:569-572).  The per-pixel steps run over
// the whole image in blocks of OBJ_CHUNK pixels or strips of up to OBJ_STRIP,
// the per-image ones in one block:
//   init, hist, thresh   range of the plane, its 1024-bin histogram, Otsu
//   strip                mask and labels of a strip of rows: 8-connected
//                        union-find in LDS; mass and coordinate sums
//   merge                unions across the strips' first rows
//   flat                 every pixel its root; Euler patterns; roots per block
//   scan, rank           rank of each root in raster order, 1-based
//   area                 areas and coordinate sums per object
//   final                distances, the two sorted lists, the features
// As one 1024-thread block per image, bound by its latency through every
// pixel, a 1388 x 1040 frame took 22 ms on one of 256 CUs.  All sums over
// pixels are of integers, so their order does not matter.
constexpr int OBJ_CHUNK = 4096;
constexpr int OBJ_STRIP = 16384;  // pixels; rows of up to 4096 pixels, so at least four rows
__host__ __device__ inline int obj_strip_rows(int W) { return OBJ_STRIP / W > 1 ? OBJ_STRIP / W : 1; }

__device__ __forceinline__ double obj_value(double v, int invert, const Stats &S) {
  return invert ? (S.mx - v) + S.mn : v;
}

__global__ void __launch_bounds__(1024) k_obj_init(const Img *imgs, const Stats *st, int invert, const ObjDesc *ods) {
  __shared__ double shd[16];
  const Img im = imgs[blockIdx.x];
  const Stats S = st[blockIdx.x];
  ObjState *T = ods[blockIdx.x].state;
  const long n = (long)im.w * im.h;
  double mn = S.mn, mx = S.mx;
  if (invert) {
    // the inversion is monotone, so its extremes are those of the extremes,
    // provided that every pixel counts (Moments2's rule) before and after
    mn = (S.mx - S.mx) + S.mn;
    mx = (S.mx - S.mn) + S.mn;
    if (S.n != n || !moments_ok(mn) || !moments_ok(mx)) {
      double a = 1e308, b = -1e308;
      for (long i = threadIdx.x; i < n; i += 1024) {
        const double v = obj_value(im.p[i], 1, S);
        if (moments_ok(v)) { a = fmin(a, v); b = fmax(b, v); }
      }
      mn = block_reduce(a, MinOp(), shd);
      mx = block_reduce(b, MaxOp(), shd);
    }
  }
  T->hist[threadIdx.x] = 0;
  if (threadIdx.x == 0) {
    T->mn = mn;
    T->mx = mx;
    T->xm = T->ym = T->mass = T->c1 = T->c3 = 0;
  }
}

__global__ void __launch_bounds__(256) k_obj_hist(const Img *imgs, const Stats *st, int invert, const ObjDesc *ods) {
  __shared__ int hist[1024];
  const Img im = imgs[blockIdx.y];
  const long n = (long)im.w * im.h, c0 = (long)blockIdx.x * OBJ_CHUNK;
  if (c0 >= n) return;
  const Stats S = st[blockIdx.y];
  ObjState *T = ods[blockIdx.y].state;
  const double mn = T->mn, sc = hist_scale(mn, T->mx, 1024);
  const gptr<const double> P = to_global((const double *)im.p);
  for (int b = threadIdx.x; b < 1024; b += 256) hist[b] = 0;
  double v[OBJ_CHUNK / 256];
#pragma unroll
  for (int k = 0; k < OBJ_CHUNK / 256; k++) v[k] = P[min(c0 + 256 * k + threadIdx.x, n - 1)];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < OBJ_CHUNK / 256; k++)
    if (c0 + 256 * k + threadIdx.x < n) atomicAdd(&hist[hist_bin(obj_value(v[k], invert, S), mn, sc, 1024)], 1);
  __syncthreads();
  for (int b = threadIdx.x; b < 1024; b += 256)
    if (hist[b]) atomicAdd(&T->hist[b], hist[b]);
}

__global__ void __launch_bounds__(1024) k_obj_thresh(const Img *imgs, const ObjDesc *ods) {
  __shared__ int hist[1024];
  const Img im = imgs[blockIdx.x];
  ObjState *T = ods[blockIdx.x].state;
  hist[threadIdx.x] = T->hist[threadIdx.x];
  __syncthreads();
  const double thr = otsu_threshold(hist, (long)im.w * im.h, T->mn, T->mx);
  if (threadIdx.x == 0) T->thr = thr;
}

__global__ void __launch_bounds__(1024) k_obj_strip(const Img *imgs, const Stats *st, int invert, const ObjDesc *ods) {
  __shared__ int lab[OBJ_STRIP];
  __shared__ long long shl[16];
  const Img im = imgs[blockIdx.y];
  const int W = im.w, RS = obj_strip_rows(W), y0 = blockIdx.x * RS;
  if (y0 >= im.h) return;
  const ObjDesc OD = ods[blockIdx.y];
  const Stats S = st[blockIdx.y];
  ObjState *T = OD.state;
  const double thr = T->thr;
  const int m = min(RS, im.h - y0) * W, base = y0 * W, t = threadIdx.x, lane = t & 63;
  const gptr<const double> P = to_global((const double *)im.p) + base;
  // A wave takes 64 consecutive pixels (raster order); each mask pixel starts
  // at the first pixel of its run inside that segment (a ballot), so runs need
  // no unions within a segment and the trees stay shallow.
  long long xm = 0, ym = 0, mass = 0;
  for (int c0 = 0; c0 < m; c0 += 4096) {
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = P[min(c0 + 1024 * k + t, m - 1)];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int i = c0 + 1024 * k + t;
      const bool in = i < m && obj_value(v[k], invert, S) > thr;
      const int y = i / W, x = i - y * W;
      // bit l: pixel l of the segment continues the run of pixel l - 1 (both
      // in the mask, the same row)
      const unsigned long long mb = __ballot(in);
      const unsigned long long cont = __ballot(in && x > 0) & (mb << 1);
      const unsigned long long below = lane == 63 ? ~0ull : ((2ull << lane) - 1);
      const int head = 63 - __clzll(~cont & below);
      if (i < m) lab[i] = in ? i - (lane - head) : -1;
      if (in) {
        xm += x + 1;
        ym += y0 + y + 1;
        mass++;
      }
    }
  }
  __syncthreads();
  // Of a horizontal run [s, e] the upper neighbours are s-1 .. e+1: each pixel
  // joins its upper-right one, the run's first pixel also its upper-left and
  // upper ones; a segment's first pixel joins its left neighbour when the run
  // crosses the segment boundary.
  auto find = [&](int x) { return uf_find(lab, x); };
  for (int i = t; i < m; i += 1024) {
    if (lab[i] < 0) continue;
    const int y = i / W, x = i - y * W;
    const bool left = x > 0 && lab[i - 1] >= 0;
    if (left && (i & 63) == 0) uf_union(lab, i, i - 1, find);
    if (y > 0) {
      const int u = i - W;
      if (x < W - 1 && lab[u + 1] >= 0) uf_union(lab, i, u + 1, find);
      if (!left) {
        if (x > 0 && lab[u - 1] >= 0) uf_union(lab, i, u - 1, find);
        if (lab[u] >= 0) uf_union(lab, i, u, find);
      }
    }
  }
  __syncthreads();
  for (int i = t; i < m; i += 1024) OD.label[base + i] = lab[i] >= 0 ? base + uf_find(lab, i) : -1;
  xm = block_reduce(xm, SumOp(), shl);
  ym = block_reduce(ym, SumOp(), shl);
  mass = block_reduce(mass, SumOp(), shl);
  if (t == 0 && mass) {
    atomicAdd((unsigned long long *)&T->xm, (unsigned long long)xm);
    atomicAdd((unsigned long long *)&T->ym, (unsigned long long)ym);
    atomicAdd((unsigned long long *)&T->mass, (unsigned long long)mass);
  }
}

__global__ void __launch_bounds__(256) k_obj_merge(const Img *imgs, const ObjDesc *ods) {
  const Img im = imgs[blockIdx.y];
  const int W = im.w, y = (blockIdx.x + 1) * obj_strip_rows(W);
  if (y >= im.h) return;
  int *lab = ods[blockIdx.y].label;
  // a label's sign never changes, so plain reads tell the mask
  auto find = [&](int x) { return uf_find_device(lab, x); };
  for (int x = threadIdx.x; x < W; x += 256) {
    const int i = y * W + x, u = i - W;
    if (lab[i] < 0) continue;
    const bool left = x > 0 && lab[i - 1] >= 0;
    if (x < W - 1 && lab[u + 1] >= 0) uf_union(lab, i, u + 1, find);
    if (!left) {
      if (x > 0 && lab[u - 1] >= 0) uf_union(lab, i, u - 1, find);
      if (lab[u] >= 0) uf_union(lab, i, u, find);
    }
  }
}

__global__ void __launch_bounds__(1024) k_obj_flat(const Img *imgs, const ObjDesc *ods) {
  __shared__ long long shl[16];
  const Img im = imgs[blockIdx.y];
  const int W = im.w, n = W * im.h, c0 = blockIdx.x * OBJ_CHUNK;
  if (c0 >= n) return;
  const ObjDesc OD = ods[blockIdx.y];
  int *lab = OD.label;
  long long c1 = 0, c3 = 0, roots = 0;
#pragma unroll
  for (int k = 0; k < OBJ_CHUNK / 1024; k++) {
    const int i = c0 + 1024 * k + threadIdx.x;
    if (i >= n) break;
    const int y = i / W, x = i - y * W;
    const int p = lab[i];
    if (y >= 1 && x >= 1) {  // EulerNumber(8): (C1 - C3) / 4; Cd is never counted
      const int c = (lab[i - W - 1] >= 0) + (lab[i - W] >= 0) + (lab[i - 1] >= 0) + (p >= 0);
      c1 += (c == 1);
      c3 += (c == 3);
    }
    if (p >= 0) {  // other threads shorten the chain meanwhile: any read of it leads to the root
      const int r = uf_find(lab, p);
      if (r != p) lab[i] = r;
      roots += r == i;
    }
  }
  c1 = block_reduce(c1, SumOp(), shl);
  c3 = block_reduce(c3, SumOp(), shl);
  roots = block_reduce(roots, SumOp(), shl);
  if (threadIdx.x == 0) {
    OD.chunk[blockIdx.x] = (int)roots;
    if (c1) atomicAdd((unsigned long long *)&OD.state->c1, (unsigned long long)c1);
    if (c3) atomicAdd((unsigned long long *)&OD.state->c3, (unsigned long long)c3);
  }
}

// exclusive prefix of the blocks' root counts
__global__ void __launch_bounds__(1024) k_obj_scan(const Img *imgs, const ObjDesc *ods) {
  __shared__ int sh[1024];
  const Img im = imgs[blockIdx.x];
  const ObjDesc OD = ods[blockIdx.x];
  const int nc = (int)(((long)im.w * im.h + OBJ_CHUNK - 1) / OBJ_CHUNK), t = threadIdx.x;
  const int per = (nc + 1023) / 1024;
  int s = 0;
  for (int k = 0; k < per; k++)
    if (t * per + k < nc) s += OD.chunk[t * per + k];
  sh[t] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int v = t >= o ? sh[t - o] : 0;
    __syncthreads();
    sh[t] += v;
    __syncthreads();
  }
  int acc = sh[t] - s;
  for (int k = 0; k < per; k++)
    if (t * per + k < nc) {
      const int c = OD.chunk[t * per + k];
      OD.chunk[t * per + k] = acc;
      acc += c;
    }
  if (t == 1023) OD.count[0] = sh[1023];
}

// label ids: rank of each root in raster order (1-based), in the sort buffer;
// the per-object sums cleared
__global__ void __launch_bounds__(1024) k_obj_rank(const Img *imgs, const ObjDesc *ods) {
  __shared__ int scan_w[16];
  const Img im = imgs[blockIdx.y];
  const int n = im.w * im.h, c0 = blockIdx.x * OBJ_CHUNK, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (c0 >= n) return;
  const ObjDesc OD = ods[blockIdx.y];
  int *rid = (int *)OD.keys;
  const int count = OD.count[0], last = c0 + OBJ_CHUNK >= n;
  int base = OD.chunk[blockIdx.x];
  for (int k = 0; k < OBJ_CHUNK / 1024; k++) {
    const int i = c0 + 1024 * k + threadIdx.x;
    const int isroot = i < n && OD.label[i] == i;
    const unsigned long long bal = __ballot(isroot);
    const int pre = __popcll(bal & ((1ull << lane) - 1));
    __syncthreads();
    if (lane == 0) scan_w[wv] = __popcll(bal);
    __syncthreads();
    int woff = 0, tot = 0;
    for (int w = 0; w < 16; w++) {
      if (w < wv) woff += scan_w[w];
      tot += scan_w[w];
    }
    if (isroot) rid[i] = base + woff + pre + 1;
    base += tot;
  }
  for (int l = c0 + threadIdx.x; l < (last ? count + 1 : min(c0 + OBJ_CHUNK, count + 1)); l += 1024) {
    OD.area[l] = 0;
    OD.xm[l] = 0;
    OD.ym[l] = 0;
  }
}

// areas and coordinate sums per object: the lanes of a wave holding one label
// add theirs first, then one lane adds the totals (exact integers)
__global__ void __launch_bounds__(1024) k_obj_area(const Img *imgs, const ObjDesc *ods) {
  const Img im = imgs[blockIdx.y];
  const int W = im.w, n = W * im.h, c0 = blockIdx.x * OBJ_CHUNK, lane = threadIdx.x & 63;
  if (c0 >= n) return;
  const ObjDesc OD = ods[blockIdx.y];
  const int *rid = (const int *)OD.keys;
  int r[OBJ_CHUNK / 1024], id[OBJ_CHUNK / 1024];
#pragma unroll
  for (int k = 0; k < OBJ_CHUNK / 1024; k++) {
    const int i = c0 + 1024 * k + threadIdx.x;
    r[k] = i < n ? OD.label[i] : -1;
  }
#pragma unroll
  for (int k = 0; k < OBJ_CHUNK / 1024; k++) id[k] = r[k] >= 0 ? rid[r[k]] : -1;
#pragma unroll
  for (int k = 0; k < OBJ_CHUNK / 1024; k++) {
    const int i = c0 + 1024 * k + threadIdx.x, l = id[k];
    const int y = i / W, x = i - y * W;
    const int px = l >= 0 ? x + 1 : 0, py = l >= 0 ? y + 1 : 0;
    for (unsigned long long pend = __ballot(l >= 0); pend;) {
      const int lead = __ffsll((long long)pend) - 1;
      const int ll = __shfl(l, lead, 64);
      const bool mine = l == ll;
      const unsigned long long mm = __ballot(mine);
      int sx = mine ? px : 0, sy = mine ? py : 0;  // at most 64 x 4096
      for (int off = 32; off > 0; off >>= 1) {
        sx += __shfl_xor(sx, off, 64);
        sy += __shfl_xor(sy, off, 64);
      }
      if (lane == lead) {
        atomicAdd(&OD.area[ll], (int)__popcll(mm));
        atomicAdd((unsigned long long *)&OD.xm[ll], (unsigned long long)sx);
        atomicAdd((unsigned long long *)&OD.ym[ll], (unsigned long long)sy);
      }
      pend &= ~mm;
    }
  }
}

__global__ void __launch_bounds__(1024) k_obj_final(const ObjDesc *ods, OutRef o) {
  __shared__ int hist[20];
  __shared__ double shd[16];
  const ObjDesc OD = ods[blockIdx.x];
  const ObjState &T = *OD.state;
  const int t = threadIdx.x, count = OD.count[0];
  const long long xm = T.xm, ym = T.ym, mass = T.mass, c1 = T.c1, c3 = T.c3;
  int *area = OD.area;
  const long long *axm = OD.xm, *aym = OD.ym;
  // per-object distance to the global centroid
  double cx = 0, cy = 0;
  if (mass) { cx = (double)xm / (double)mass; cy = (double)ym / (double)mass; }
  uint64_t *ka = OD.keys, *kb = OD.keys + (count + 1);
  double *dist = OD.dist;
  double sum_d = 0;
  for (long l = t; l < count; l += 1024) {
    const long L = l + 1;
    const double xc = (double)axm[L] / (double)area[L], yc = (double)aym[L] / (double)area[L];
    const double dx = xc - cx, dy = yc - cy;
    const double d = sqrt(dx * dx + dy * dy);
    dist[l] = d;
    sum_d += d;
  }
  sum_d = block_reduce(sum_d, SumOp(), shd);
  // sort the areas (as integer keys)
  for (long l = t; l < count; l += 1024) ka[l] = (uint64_t)area[l + 1];
  __syncthreads();
  uint64_t *sa = block_radix_sort(ka, kb, count);
  // sorted areas -> dist buffer tail? keep them in place: copy to area[] (1-based free now)
  for (long l = t; l < count; l += 1024) area[l] = (int)sa[l];
  __syncthreads();
  for (long l = t; l < count; l += 1024) ka[l] = dkey(dist[l]);
  __syncthreads();
  uint64_t *sd = block_radix_sort(ka, kb, count);
  for (long l = t; l < count; l += 1024) dist[l] = dkey_inv(sd[l]);
  __syncthreads();
  // statistics (count == 0 reads an empty array in the reference; defined as 0 here)
  const double sum_a = (double)mass;  // sum of object areas == mask pixel count
  double AreaMean = 0, DistMean = 0, amin = 0, amax = 0, dmin = 0, dmax = 0;
  if (count > 0) {
    amin = area[0]; amax = area[count - 1];
    dmin = dist[0]; dmax = dist[count - 1];
    AreaMean = sum_a / count;
    DistMean = sum_d / count;
  }
  if (t < 20) hist[t] = 0;
  __syncthreads();
  double va = 0, vd = 0;
  const double hsa = (amax - amin > 0) ? 10.0 / (double)(amax - amin) : 0.0;
  const double hsd = (dmax - dmin > 0) ? 10.0 / (double)(dmax - dmin) : 0.0;
  for (long l = t; l < count; l += 1024) {
    if (amax - amin > 0) {
      const double da = area[l] - AreaMean;
      va += da * da;
      atomicAdd(&hist[hist_bin((double)area[l], amin, hsa, 10)], 1);
    }
    const double dd = dist[l] - DistMean;
    vd += dd * dd;
    atomicAdd(&hist[10 + hist_bin(dist[l], dmin, hsd, 10)], 1);
  }
  va = block_reduce(va, SumOp(), shd);
  vd = block_reduce(vd, SumOp(), shd);
  if (t == 0) {
    double *out = o.rows[blockIdx.x];
    int k = 0;
    for (int j = 0; j < 10; j++) out[k++] = hist[j];
    out[k++] = amax;
    out[k++] = AreaMean;
    out[k++] = count > 0 ? (double)(unsigned)area[count / 2] : 0.0;
    out[k++] = amin;
    out[k++] = count > 1 ? va / (count - 1) : va;
    out[k++] = cx;
    out[k++] = cy;
    out[k++] = count;
    for (int j = 0; j < 10; j++) out[k++] = hist[10 + j];
    out[k++] = dmax;
    out[k++] = DistMean;
    out[k++] = count > 0 ? dist[count / 2] : 0.0;
    out[k++] = dmin;
    out[k++] = count > 1 ? vd / (count - 1) : vd;
    out[k++] = (double)((c1 - c3) / 4);
  }
}

// Images or planes of a launch whose grid has them in y, which by the device's
// limits takes up to 65,536: a call may have more (edge features two planes per
// image, the object features one per node of the plan), so these launches go in
// slices.
constexpr int GRID_Y = 65536;
template <class Launch>
static void in_slices(int n, Launch launch) {
  for (int i = 0; i < n; i += GRID_Y) launch(i, std::min(n - i, GRID_Y));
}

void launch_objects(const Img *imgs, const Stats *st, int invert, const ObjDesc *od, OutRef o, int nimg, long maxn,
                    int maxstrips, hipStream_t s) {
  in_slices(nimg, [&](int i, int n) {
    const Img *im = imgs + i;
    const ObjDesc *d = od + i;
    const dim3 chunks((unsigned)((maxn + OBJ_CHUNK - 1) / OBJ_CHUNK), n);
    k_obj_init<<<n, 1024, 0, s>>>(im, st + i, invert, d);
    k_obj_hist<<<chunks, 256, 0, s>>>(im, st + i, invert, d);
    k_obj_thresh<<<n, 1024, 0, s>>>(im, d);
    k_obj_strip<<<dim3(maxstrips, n), 1024, 0, s>>>(im, st + i, invert, d);
    if (maxstrips > 1) k_obj_merge<<<dim3(maxstrips - 1, n), 256, 0, s>>>(im, d);
    k_obj_flat<<<chunks, 1024, 0, s>>>(im, d);
    k_obj_scan<<<n, 1024, 0, s>>>(im, d);
    k_obj_rank<<<chunks, 1024, 0, s>>>(im, d);
    k_obj_area<<<chunks, 1024, 0, s>>>(im, d);
    k_obj_final<<<n, 1024, 0, s>>>(d, OutRef{o.rows + i});
  });
}
int obj_strips(int h, int w) { return (h + obj_strip_rows(w) - 1) / obj_strip_rows(w); }
int obj_chunks(long n) { return (int)((n + OBJ_CHUNK - 1) / OBJ_CHUNK); }

// ================================================================ Edge features
// Prewitt magnitude / direction (cmatrix.cpp:1317-1384), x outer order of the
// reference is irrelevant per pixel; the accumulation order inside a pixel is kept.
__global__ void k_prewitt(const Img *in, const Img *mag, const Img *dir) {
  const Img a = in[blockIdx.y], om = mag[blockIdx.y], od = dir[blockIdx.y];
  const long w = a.w, h = a.h;
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= w * h) return;
  const long y = i / w, x = i - y * w;
  double sumx = 0, sumy = 0;
  for (long j = y - 1; j <= y + 1; j++) if (j >= 0 && j < h && x - 1 >= 0) sumx += a.p[j * w + x - 1] * 1;
  for (long j = y - 1; j <= y + 1; j++) if (j >= 0 && j < h && x + 1 < w) sumx += a.p[j * w + x + 1] * -1;
  for (long k = x - 1; k <= x + 1; k++) if (k >= 0 && k < w && y - 1 >= 0) sumy += a.p[(y - 1) * w + k] * 1;
  for (long k = x - 1; k <= x + 1; k++) if (k >= 0 && k < w && y + 1 < h) sumy += a.p[(y + 1) * w + k] * -1;
  om.p[i] = sqrt(sumx * sumx + sumy * sumy);
  double d;
  if (sumy == 0 || fabs(sumy) < 1 / kInf) d = 3.1415926 * (sumx < 0 ? 1 : 0);
  else d = atan2(sumy, sumx);
  od.p[i] = d;
}

// ------------------------------------------------------------------ medians
// Median of each plane (ImageMatrix::get_median, cmatrix.cpp:780-800) without
// sorting it: the values are counted in SEL_BINS bins between the plane's
// extremes (a binning that follows the keys' order, NaN and infinities
// included), the keys of the bin or two that hold the middle ranks are
// collected, and one block finds the ranks among those, digit by digit.  A
// 1388 x 1040 frame's two edge planes took 17 of 20.8 ms as one-block radix
// sorts.
__device__ __forceinline__ int sel_bin(double v, double mn, double mx, double scale) {
  if (v != v) return __double_as_longlong(v) < 0 ? 0 : SEL_BINS - 1;
  if (v <= mn) return 0;
  if (v >= mx) return SEL_BINS - 1;
  return min((int)((v - mn) * scale), SEL_BINS - 1);
}
__global__ void __launch_bounds__(1024) k_sel_init(SelState *sel) {
  SelState &T = sel[blockIdx.x];
  for (int b = threadIdx.x; b < SEL_BINS; b += 1024) T.hist[b] = 0;
  if (threadIdx.x == 0) {
    T.count = 0;
    T.kmin = ~0ull;
    T.kmax = 0;
  }
}
__global__ void __launch_bounds__(256) k_sel_hist(const Img *planes, const Stats *st, SelState *sel) {
  __shared__ int hist[SEL_BINS];
  const Img im = planes[blockIdx.y];
  const long n = (long)im.w * im.h, c0 = (long)blockIdx.x * SEL_CHUNK;
  if (c0 >= n) return;
  const Stats S = st[blockIdx.y];
  SelState &T = sel[blockIdx.y];
  const double scale = hist_scale(S.mn, S.mx, SEL_BINS);
  const gptr<const double> P = to_global((const double *)im.p);
  for (int b = threadIdx.x; b < SEL_BINS; b += 256) hist[b] = 0;
  __syncthreads();
  for (int r = 0; r < SEL_CHUNK; r += 256 * 16) {
    double v[16];
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = P[min(c0 + r + 256 * k + threadIdx.x, n - 1)];
#pragma unroll
    for (int k = 0; k < 16; k++)
      if (c0 + r + 256 * k + threadIdx.x < n) atomicAdd(&hist[sel_bin(v[k], S.mn, S.mx, scale)], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < SEL_BINS; b += 256)
    if (hist[b]) atomicAdd(&T.hist[b], hist[b]);
}
// the bins of ranks (n - 1) / 2 and n / 2
__global__ void __launch_bounds__(1024) k_sel_pick(const Img *planes, SelState *sel) {
  __shared__ int sh[1024];
  const Img im = planes[blockIdx.x];
  const int n = im.w * im.h, t = threadIdx.x, r0 = (n - 1) / 2, r1 = n / 2;
  SelState &T = sel[blockIdx.x];
  constexpr int PER = SEL_BINS / 1024;
  int c[PER], s = 0;
#pragma unroll
  for (int k = 0; k < PER; k++) s += c[k] = T.hist[t * PER + k];
  sh[t] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int v = t >= o ? sh[t - o] : 0;
    __syncthreads();
    sh[t] += v;
    __syncthreads();
  }
  int acc = sh[t] - s;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    if (r0 >= acc && r0 < acc + c[k]) {
      T.lo = t * PER + k;
      T.rank = r0 - acc;
    }
    if (r1 >= acc && r1 < acc + c[k]) T.hi = t * PER + k;
    acc += c[k];
  }
}
__global__ void __launch_bounds__(256) k_sel_collect(const Img *planes, const Stats *st, SelState *sel, uint64_t *const *keys) {
  const Img im = planes[blockIdx.y];
  const long n = (long)im.w * im.h, c0 = (long)blockIdx.x * SEL_CHUNK;
  if (c0 >= n) return;
  const Stats S = st[blockIdx.y];
  SelState &T = sel[blockIdx.y];
  uint64_t *out = keys[blockIdx.y];
  const int lo = T.lo, hi = T.hi, lane = threadIdx.x & 63;
  const double scale = hist_scale(S.mn, S.mx, SEL_BINS);
  const gptr<const double> P = to_global((const double *)im.p);
  uint64_t kmin = ~0ull, kmax = 0;
  for (int r = 0; r < SEL_CHUNK; r += 256 * 16) {
    double v[16];
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = P[min(c0 + r + 256 * k + threadIdx.x, n - 1)];
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const int b = sel_bin(v[k], S.mn, S.mx, scale);
      const bool in = c0 + r + 256 * k + threadIdx.x < n && (b == lo || b == hi);
      const unsigned long long m = __ballot(in);
      if (m == 0) continue;
      int base = 0;
      if (lane == 0) base = atomicAdd(&T.count, (int)__popcll(m));
      base = __shfl(base, 0, 64);
      if (in) {
        const uint64_t key = dkey(v[k]);
        out[base + __popcll(m & ((1ull << lane) - 1))] = key;
        kmin = key < kmin ? key : kmin;
        kmax = key > kmax ? key : kmax;
      }
    }
  }
  if (kmin <= kmax) {
    atomicMin((unsigned long long *)&T.kmin, (unsigned long long)kmin);
    atomicMax((unsigned long long *)&T.kmax, (unsigned long long)kmax);
  }
}
__global__ void __launch_bounds__(1024) k_sel_final(const Img *planes, const SelState *sel, uint64_t *const *keys, double *median) {
  __shared__ int hist[256];
  __shared__ unsigned long long s_next;
  __shared__ int s_digit, s_rank;
  const Img im = planes[blockIdx.x];
  const SelState &T = sel[blockIdx.x];
  const int n = im.w * im.h, m = T.count, t = threadIdx.x;
  const uint64_t *k = keys[blockIdx.x];
  uint64_t k0 = T.kmin, k1 = T.kmin;
  if (T.kmin != T.kmax) {
    // the key of rank T.rank: its digits from the highest, the keys that share
    // the digits found so far counted by the next one
    uint64_t prefix = 0, mask = 0;
    int rank = T.rank, equal = 0;
    for (int sh = 56; sh >= 0; sh -= 8) {
      if (((T.kmin ^ T.kmax) >> sh) == 0) {  // a leading part that all keys share
        mask |= 0xffull << sh;
        prefix |= T.kmin & (0xffull << sh);
        equal = m;
        continue;
      }
      for (int b = t; b < 256; b += 1024) hist[b] = 0;
      __syncthreads();
      for (int i = t; i < m; i += 1024)
        if ((k[i] & mask) == prefix) atomicAdd(&hist[(k[i] >> sh) & 255], 1);
      __syncthreads();
      if (t == 0) {
        int b = 0, r = rank;
        while (r >= hist[b]) r -= hist[b++];
        s_digit = b;
        s_rank = r;
      }
      __syncthreads();
      rank = s_rank;
      equal = hist[s_digit];
      prefix |= (uint64_t)s_digit << sh;
      mask |= 0xffull << sh;
      __syncthreads();
    }
    k0 = k1 = prefix;
    if (n % 2 == 0 && rank + 1 >= equal) {  // the next rank is the smallest larger key
      if (t == 0) s_next = ~0ull;
      __syncthreads();
      uint64_t best = ~0ull;
      for (int i = t; i < m; i += 1024)
        if (k[i] > k0 && k[i] < best) best = k[i];
      if (best != ~0ull) atomicMin(&s_next, (unsigned long long)best);
      __syncthreads();
      k1 = s_next;
    }
  }
  if (t == 0) {
    double med;
    if (n % 2 == 0) {
      med = dkey_inv(k1);
      med += dkey_inv(k0);
      med /= 2.0;
    } else {
      med = dkey_inv(k0);
    }
    median[blockIdx.x] = med;
  }
}

// EdgeStatistics (cmatrix.cpp:1402-1458) + output layout (FeatureAlgorithms.cpp:314-335).
// st2[2*i] / st2[2*i+1] and medians[2*i] / [2*i+1] belong to magnitude / direction.
// Counts over blocks of pixels: each thread counts its own pixels' bins in the
// bytes of two words, then the wave and the block add them.
__global__ void __launch_bounds__(256) k_edge_count(const Img *mag, const Img *dir, const Stats *st2, EdgeCounts *cnt) {
  const Img M = mag[blockIdx.y], D = dir[blockIdx.y];
  const long n = (long)M.h * M.w, c0 = (long)blockIdx.x * SEL_CHUNK;
  if (c0 >= n) return;
  const Stats SM = st2[2 * blockIdx.y], SD = st2[2 * blockIdx.y + 1];
  const double level = SM.mean;
  const double sm = hist_scale(SM.mn, SM.mx, 8), sd = hist_scale(SD.mn, SD.mx, 8);
  const gptr<const double> PM = to_global((const double *)M.p), PD = to_global((const double *)D.p);
  static_assert(SEL_CHUNK / 256 < 256, "a thread's pixels are counted in bytes");
  uint64_t wm = 0, wd = 0;
  int area = 0;
  for (int r = 0; r < SEL_CHUNK; r += 256 * 8) {
    double a[8], b[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const long i = min(c0 + r + 256 * k + threadIdx.x, n - 1);
      a[k] = PM[i];
      b[k] = PD[i];
    }
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (c0 + r + 256 * k + threadIdx.x < n) {
        area += a[k] > level;
        wm += 1ull << (8 * hist_bin(a[k], SM.mn, sm, 8));
        wd += 1ull << (8 * hist_bin(b[k], SD.mn, sd, 8));
      }
  }
  EdgeCounts &T = cnt[blockIdx.y];
  auto add = [&](int v, int *p) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0 && v) atomicAdd(p, v);
  };
  add(area, &T.area);
#pragma unroll
  for (int b = 0; b < 8; b++) {
    add((int)((wm >> (8 * b)) & 255), &T.hm[b]);
    add((int)((wd >> (8 * b)) & 255), &T.hd[b]);
  }
}
__global__ void __launch_bounds__(64) k_edge_final(const EdgeCounts *cnt, const Stats *st2, const double *medians, OutRef o) {
  if (threadIdx.x != 0) return;
  const Stats SM = st2[2 * blockIdx.x], SD = st2[2 * blockIdx.x + 1];
  const EdgeCounts &T = cnt[blockIdx.x];
  double DH[8], MH[8], diff[4] = {0, 0, 0, 0}, homog = 0;
  for (int b = 0; b < 8; b++) { DH[b] = T.hd[b]; MH[b] = T.hm[b]; }
  for (int b = 0; b < 4; b++) diff[b] = fabs(DH[b] - DH[b + 4]);
  double sum = 0;
  for (int b = 0; b < 4; b++) {
    if (DH[b] + DH[b + 4] != 0) diff[b] = diff[b] / (DH[b] + DH[b + 4]);
    sum += (DH[b] + DH[b + 4]);
  }
  if (sum > 0) homog = (DH[0] + DH[1]) / sum;
  double *c = o.rows[blockIdx.x];
  int h = 0;
  c[h++] = (double)T.area;
  for (int j = 0; j < 4; j++) c[h++] = diff[j];
  for (int j = 0; j < 8; j++) c[h++] = DH[j];
  c[h++] = homog;
  c[h++] = SD.mean;
  c[h++] = medians[2 * blockIdx.x + 1];
  c[h++] = SD.var;
  for (int j = 0; j < 8; j++) c[h++] = MH[j];
  c[h++] = SM.mean;
  c[h++] = medians[2 * blockIdx.x];
  c[h++] = SM.var;
}

void launch_median(const Img *planes, const Stats *st, SelState *sel, uint64_t *const *keys, double *median, int nplanes,
                   long maxn, hipStream_t s) {
  in_slices(nplanes, [&](int i, int n) {
    const dim3 chunks((unsigned)((maxn + SEL_CHUNK - 1) / SEL_CHUNK), n);
    k_sel_init<<<n, 1024, 0, s>>>(sel + i);
    k_sel_hist<<<chunks, 256, 0, s>>>(planes + i, st + i, sel + i);
    k_sel_pick<<<n, 1024, 0, s>>>(planes + i, sel + i);
    k_sel_collect<<<chunks, 256, 0, s>>>(planes + i, st + i, sel + i, keys + i);
    k_sel_final<<<n, 1024, 0, s>>>(planes + i, sel + i, keys + i, median + i);
  });
}
void launch_prewitt(const Img *imgs, const Img *mag, const Img *dir, int nimg, long maxn, hipStream_t s) {
  k_prewitt<<<dim3((maxn + 255) / 256, nimg), 256, 0, s>>>(imgs, mag, dir);
}

void launch_edge_final(const Img *mag, const Img *dir, const Stats *st2, const double *medians, EdgeCounts *cnt, OutRef o,
                       int nimg, long maxn, hipStream_t s) {
  launch_fill_int((int *)cnt, (long)nimg * (long)(sizeof(EdgeCounts) / sizeof(int)), 0, s);
  k_edge_count<<<dim3((unsigned)((maxn + SEL_CHUNK - 1) / SEL_CHUNK), nimg), 256, 0, s>>>(mag, dir, st2, cnt);
  k_edge_final<<<nimg, 64, 0, s>>>(cnt, st2, medians, o);
}

// ======================================================================= Gabor
// GaborTextureFilters2D (gabor.cpp:201-231) with GaborEnergy / conv2comp
// (gabor.cpp:19-52,166-195).  kernels: 8 host-computed normalised complex
// 38x38 filters (index 0 = low-pass f0 = 0.1, 1..7 = f0 1..7).  Each output
// pixel accumulates the 1444 taps in the reference's (row, column) tap order
// with separate multiply and add; taps that fall outside the image add
// +-0, which leaves the sum unchanged.
#define GB_N 38
#define GB_TR 32          // output rows per block
#define GB_TC 64          // output columns per block
#define GB_LD (GB_TC + GB_N - 1 + 1)
// Block = 32 x 64 outputs of one filter on one image; thread = 8 adjacent
// outputs of one row.  Taps are taken in groups of eight: the 15 input values
// a group needs for the thread's 8 outputs are read from LDS once into
// registers, and every output still adds its taps in the reference's (j, i)
// order (conv2comp, gabor.cpp:19-52).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_gabor_conv(const Img *imgs, const double *kernels, double *const *energy) {
  __shared__ double tile[GB_TR + GB_N - 1][GB_LD];
  __shared__ double2 wk[GB_N * GB_N];
  const Img im = imgs[blockIdx.z];
  const int f = blockIdx.y % 8;
  const int tilesx = (im.w + GB_TC - 1) / GB_TC, tilesy = (im.h + GB_TR - 1) / GB_TR;
  if ((int)blockIdx.x >= tilesx * tilesy) return;
  const int b0 = (blockIdx.x / tilesx) * GB_TR, a0 = (blockIdx.x % tilesx) * GB_TC;
  const int t = threadIdx.x;
  const double *K = kernels + (long)f * GB_N * GB_N * 2;
  for (int e = t; e < GB_N * GB_N; e += 256) wk[e] = make_double2(K[2 * e], K[2 * e + 1]);
  // input rows b0-18 .. b0+GB_TR+18, columns a0-18 .. a0+GB_TC+18
  for (int r = t / 64; r < GB_TR + GB_N - 1; r += 4) {
    const int y = b0 - 18 + r;
    for (int c = t % 64; c < GB_TC + GB_N - 1; c += 64) {
      const int x = a0 - 18 + c;
      tile[r][c] = (y >= 0 && y < im.h && x >= 0 && x < im.w) ? im.p[(long)y * im.w + x] : 0.0;
    }
  }
  __syncthreads();
  const int ty = t / 8, tx = t % 8;
  const int b = b0 + ty, a = a0 + tx * 8;
  double re[8], imv[8];
#pragma unroll
  for (int q = 0; q < 8; q++) re[q] = imv[q] = 0.0;
  const int rb = ty + 37, cb = tx * 8 + 37;
#pragma unroll 1
  for (int j = 0; j < GB_N; j++) {
    const double *row = &tile[rb - j][0];
    const double2 *wr = &wk[j * GB_N];
#pragma unroll
    for (int i0 = 0; i0 < GB_N; i0 += 8) {
      // u[k] = row[cb - i0 - 7 + k]: value of output q, tap i is u[q - (i - i0) + 7]
      // taps in this group: D = min(8, GB_N - i0); slots k < 8 - D are unused
      const int D = (GB_N - i0 < 8) ? GB_N - i0 : 8;
      double u[15];
#pragma unroll
      for (int k = 0; k < 15; k++) u[k] = (k >= 8 - D) ? row[cb - i0 - 7 + k] : 0.0;
#pragma unroll
      for (int di = 0; di < 8; di++) {
        if (i0 + di < GB_N) {
          const double2 w = wr[i0 + di];
#pragma unroll
          for (int q = 0; q < 8; q++) {
            const double v = u[q - di + 7];
            re[q] += v * w.x;
            imv[q] += v * w.y;
          }
        }
      }
    }
  }
  double *E = energy[blockIdx.z] + (long)f * im.h * im.w;
  if (b < im.h)
#pragma unroll
    for (int q = 0; q < 8; q++)
      if (a + q < im.w) E[(long)b * im.w + a + q] = sqrt(re[q] * re[q] + imv[q] * imv[q]);
}

// The energies E with an a-priori bound D on each one's distance from
// k_gabor_conv's value E64, for launch_gabor_post_exact to certify every count
// (k_gabor_repair recomputes in k_gabor_conv's order each energy a count leaves
// open).
//
// A filter is, to 4e-16 of the sum of its taps' magnitudes, the sum of two
// products of a row and a column: w(j, i) = b0(j) a0(i) + b1(j) a1(i), a real and
// b complex, the second for the filter's angle, which is not quite pi / 2.  So
// the image is filtered along its rows twice and along its columns with two
// complex filters: 228 fused multiply-adds per energy (and 1.4 times the first
// 76, for the rows around the block's) instead of 2,888.
//
// Bound: E64's components are within gamma_1445 S of the exact sum, S =
// sum |x| |w| <= (largest |x| of the block's input tile) x wsum_f; these within
// (gamma_39 + gamma_80 + 4e-16) (1 + 1e-8) S; the magnitudes round by at most 2u
// each: |E - E64| <= 1.8e-13 S + 4u E.  D = coef * tmax * wsum_f + 1e-14 E with
// coef = 4e-13 times the context's slack, rounded up.  Where a block's largest
// |x| is so small that D would leave float's range, so large that a sum could
// overflow, or infinite, its energies are E64 itself: the 1,444 products, each
// rounded and added in k_gabor_conv's order, with D = 0.
//
// A block takes 27 x 64 outputs, i.e. 64 rows of 101 inputs, and `per` filters.
// Each of 512 threads forms eight adjacent row sums of both kinds from a sliding
// window of registers, then a wave four rows of 64 energies; the taps are uniform
// and come through the scalar cache.  400 images of 256 x 256: 6.7 ms, 21.8 ms
// with 1,444 complex taps per energy; three of 1388 x 1040: 1.2 ms, 4.6 ms.
#define GS_TR 27
#define GS_IN (GS_TR + GB_N - 1)
constexpr int GS_F = 6 * GB_N;  // factors of a filter: a0, a1, re b0, im b0, re b1, im b1
static_assert(GS_IN == 64, "eight threads per input row");
__global__ void __launch_bounds__(512) k_gabor_sep(const Img *imgs, const double *__restrict__ factors,
                                                   const double *__restrict__ kernels, double *const *energy,
                                                   const double *__restrict__ wsum, float *const *bound, double coef,
                                                   int per) {
  __shared__ double tile[GS_IN][GB_LD + 1];
  __shared__ double rows[2][GS_IN][GB_TC + 1];
  __shared__ double shd[8];
  const Img im = imgs[blockIdx.z];
  const int tilesx = (im.w + GB_TC - 1) / GB_TC, tilesy = (im.h + GS_TR - 1) / GS_TR;
  if ((int)blockIdx.x >= tilesx * tilesy) return;
  const int b0 = (blockIdx.x / tilesx) * GS_TR, a0 = (blockIdx.x % tilesx) * GB_TC;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const long plane = (long)im.h * im.w;
  // input rows b0-18 .. b0+45, columns a0-18 .. a0+82
  double tmax = 0.0;
  for (int r = wave; r < GS_IN; r += 8) {
    const int y = b0 - 18 + r;
    for (int c = lane; c < GB_TC + GB_N - 1; c += 64) {
      const int x = a0 - 18 + c;
      const double v = (y >= 0 && y < im.h && x >= 0 && x < im.w) ? im.p[(long)y * im.w + x] : 0.0;
      tile[r][c] = v;
      tmax = fmax(tmax, fabs(v));
    }
  }
  tmax = block_reduce(tmax, MaxOp(), shd);  // (synchronises the block)
  const bool sized = tmax == 0.0 || (tmax >= 1e-24 && tmax <= 1e290);
  for (int f = blockIdx.y * per; f < (int)(blockIdx.y + 1) * per; f++) {
    double *E = energy[blockIdx.z] + f * plane;
    float *D = bound[blockIdx.z] + f * plane;
    const double db = coef * tmax * wsum[f];
    auto put = [&](int y, int x, double re, double imv) {
      if (y >= im.h || x >= im.w) return;
      const double e = sqrt(re * re + imv * imv);
      E[(long)y * im.w + x] = e;
      D[(long)y * im.w + x] = (float)((db + 1e-14 * e) * 1.000001);
    };
    if (!sized) {
      const double *K = kernels + (long)f * GB_N * GB_N * 2;
      for (int r = wave; r < GS_TR; r += 8) {
        const int y = b0 + r, x = a0 + lane;
        double re = 0.0, imv = 0.0;
        for (int j = 0; j < GB_N; j++)
          for (int i = 0; i < GB_N; i++) {
            const double v = tile[r + 37 - j][lane + 37 - i];
            re += v * K[2 * (j * GB_N + i)];
            imv += v * K[2 * (j * GB_N + i) + 1];
          }
        if (y >= im.h || x >= im.w) continue;
        const double e = sqrt(re * re + imv * imv);
        E[(long)y * im.w + x] = e;
        D[(long)y * im.w + x] = e == e ? 0.0f : (float)e;  // (NaN stays undecided, as elsewhere)
      }
      continue;
    }
    const double *F = factors + f * GS_F;
    {
      const int r = t >> 3, c0 = (t & 7) * 8;
      double h0[8], h1[8];
#pragma unroll
      for (int q = 0; q < 8; q++) h0[q] = h1[q] = 0.0;
      // output c0 + q takes tap i from input column c0 + q + 37 - i
#pragma unroll
      for (int i0 = 0; i0 < GB_N; i0 += 8) {
        const int nt = GB_N - i0 < 8 ? GB_N - i0 : 8;
        double u[15];
#pragma unroll
        for (int k = 0; k < 15; k++) u[k] = k >= 8 - nt ? tile[r][c0 + 30 - i0 + k] : 0.0;
#pragma unroll
        for (int di = 0; di < nt; di++) {
          const double w0 = F[i0 + di], w1 = F[GB_N + i0 + di];
#pragma unroll
          for (int q = 0; q < 8; q++) {
            h0[q] = fma(u[q - di + 7], w0, h0[q]);
            h1[q] = fma(u[q - di + 7], w1, h1[q]);
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 8; q++) {
        rows[0][r][c0 + q] = h0[q];
        rows[1][r][c0 + q] = h1[q];
      }
    }
    __syncthreads();
    if (wave * 4 < GS_TR) {
      double re[4] = {0, 0, 0, 0}, imv[4] = {0, 0, 0, 0};
      const int r0 = wave * 4;  // output r0 + q takes tap j from row r0 + q + 37 - j
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const double *B = F + (2 + 2 * p) * GB_N;
#pragma unroll
        for (int j0 = 0; j0 < GB_N; j0 += 8) {
          const int nt = GB_N - j0 < 8 ? GB_N - j0 : 8;
          double u[11];
#pragma unroll
          for (int k = 0; k < 11; k++) u[k] = k >= 8 - nt ? rows[p][min(r0 + 30 - j0 + k, GS_IN - 1)][lane] : 0.0;
#pragma unroll
          for (int dj = 0; dj < nt; dj++) {
            const double wr = B[j0 + dj], wi = B[GB_N + j0 + dj];
#pragma unroll
            for (int q = 0; q < 4; q++) {
              re[q] = fma(u[q - dj + 7], wr, re[q]);
              imv[q] = fma(u[q - dj + 7], wi, imv[q]);
            }
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (r0 + q < GS_TR) put(b0 + r0 + q, a0 + lane, re[q], imv[q]);
    }
    __syncthreads();  // the next filter's row sums overwrite these
  }
}

__global__ void __launch_bounds__(1024) k_gabor_post(const Img *imgs, double *const *energy, OutRef o) {
  __shared__ int hist[1024];
  __shared__ double shd[16];
  __shared__ long long shl[16];
  const Img im = imgs[blockIdx.x];
  const long n = (long)im.h * im.w;
  const double *E0 = energy[blockIdx.x];
  double *out = o.rows[blockIdx.x];
  long long orig = 0;
  for (int f = 0; f < 8; f++) {
    const double *E = E0 + (long)f * n;
    // (the per-pixel loops are unrolled so that four loads are in flight)
    double mx = -1e308;
#pragma unroll 4
    for (long i = threadIdx.x; i < n; i += 1024) mx = fmax(mx, E[i]);
    mx = block_reduce(mx, MaxOp(), shd);
    if (f == 0) {
      long long c = 0;
      const double lvl = mx * 0.4;
#pragma unroll 4
      for (long i = threadIdx.x; i < n; i += 1024) c += E[i] > lvl;
      orig = block_reduce(c, SumOp(), shl);
      continue;
    }
    // e / max, its min / max, Otsu threshold, count above
    double a = 1e308, b = -1e308;
#pragma unroll 4
    for (long i = threadIdx.x; i < n; i += 1024) {
      const double v = E[i] / mx;
      if (moments_ok(v)) { a = fmin(a, v); b = fmax(b, v); }
    }
    a = block_reduce(a, MinOp(), shd);
    b = block_reduce(b, MaxOp(), shd);
    const double thr = block_otsu(n, a, b, [&](long i) { return E[i] / mx; }, hist);
    long long c = 0;
#pragma unroll 4
    for (long i = threadIdx.x; i < n; i += 1024) c += (E[i] / mx) > thr;
    c = block_reduce(c, SumOp(), shl);
    if (threadIdx.x == 0) out[f - 1] = (double)c / (double)orig;
  }
}

// The Gabor ratios from energies E with bounds D (|E - E64| <= D, E64 =
// k_gabor_conv's value: the fused multiply-add, FP32 and BF16
// forms), equal to k_gabor_post on the FP64 energies.  Every decision whose
// interval [E - D, E + D] leaves it open is taken on E64: the pixels
// concerned are marked (D < 0), and the repairs recompute them in
// k_gabor_conv's tap order (E = E64, D = 0).  Five phases of
// launch_gabor_post_exact, each followed by the repairs except the last:
//   1  mark the candidates for the maximum (upper end >= largest lower end)
//   2  max M; filter 0: mark the pixels open at 0.4 M; other filters: mark
//      the candidates for the minimum of e / M
//   3  filter 0: the base count; others: min a and max b of e / M, mark the
//      pixels whose Otsu bin is open
//   4  Otsu histogram and threshold; mark the pixels open at the threshold
//   5  the counts above the threshold, the ratios

// the marked pixels (D < 0) of one 32 x 64 tile of one filter's map: the
// input window staged in LDS as k_gabor_conv does, each marked output then
// summed in k_gabor_conv's tap order by one lane
__device__ void gabor_repair_tile(const Img &im, int tile, const double *K, double *E, float *D,
                                  double (*tile_px)[GB_LD], double2 *wk, int *list, int *nlist) {
  const int tilesx = (im.w + GB_TC - 1) / GB_TC;
  const int b0 = (tile / tilesx) * GB_TR, a0 = (tile % tilesx) * GB_TC;
  const int t = threadIdx.x;
  if (t == 0) *nlist = 0;
  __syncthreads();
  for (int e = t; e < GB_TR * GB_TC; e += 256) {
    const int r = e / GB_TC, c = e - r * GB_TC;
    const int y = b0 + r, x = a0 + c;
    if (y < im.h && x < im.w && D[(long)y * im.w + x] < 0.0f) list[atomicAdd(nlist, 1)] = e;
  }
  __syncthreads();
  const int nl = *nlist;
  if (nl == 0) return;  // (uniform: every thread returns)
  for (int e = t; e < GB_N * GB_N; e += 256) wk[e] = make_double2(K[2 * e], K[2 * e + 1]);
  for (int r = t / 64; r < GB_TR + GB_N - 1; r += 4) {
    const int y = b0 - 18 + r;
    for (int c = t % 64; c < GB_TC + GB_N - 1; c += 64) {
      const int x = a0 - 18 + c;
      tile_px[r][c] = (y >= 0 && y < im.h && x >= 0 && x < im.w) ? im.p[(long)y * im.w + x] : 0.0;
    }
  }
  __syncthreads();
  for (int k = t; k < nl; k += 256) {
    const int e = list[k];
    const int r = e / GB_TC, c = e - r * GB_TC;
    // output (b0 + r, a0 + c) reads tile row r + 37 - j, column c + 37 - i
    double re = 0.0, imv = 0.0;
    for (int j = 0; j < GB_N; j++) {
      const double *row = &tile_px[r + 37 - j][c + 37];
      const double2 *wr = &wk[j * GB_N];
#pragma unroll
      for (int i = 0; i < GB_N; i++) {
        const double v = row[-i];
        const double2 w = wr[i];
        re += v * w.x;
        imv += v * w.y;
      }
    }
    const long o = (long)(b0 + r) * im.w + a0 + c;
    E[o] = sqrt(re * re + imv * imv);
    D[o] = 0.0f;
  }
  __syncthreads();  // the buffers are reused by the next tile
}

// Per (image, filter), flags[(8 image + filter) * GR_STRIDE] holds the
// number of energies the last phase marked there and, when at most GR_CAP,
// their pixel indices.  k_gabor_repair_list recomputes listed energies one
// per thread straight from global memory; k_gabor_repair takes the filters
// with more, tile by tile.  Grid (tiles, 8, images), one tile per block, or
// (1, 8, images) with each block taking its filter's tiles in turn
// (loop_tiles: for bounds that leave few energies open).
constexpr int GR_CAP = 63;
constexpr int GR_STRIDE = GR_CAP + 1;
// One wavefront per (image, filter); per listed energy the lanes form the
// 1444 tap products (each rounded once, as in the sum) into LDS, and lane 0
// adds them in k_gabor_conv's (and the tile repair's) order: tap
// (j, i) reads input (y + 19 - j, x + 19 - i), +0 outside the image.
__global__ void __launch_bounds__(64) k_gabor_repair_list(const Img *imgs, const double *kernels, double *const *energy,
                                                          float *const *bound, const int *flags) {
  __shared__ double pre[GB_N * GB_N], pim[GB_N * GB_N];
  const int f = blockIdx.y;
  const int *fl = flags + (long)(blockIdx.z * 8 + f) * GR_STRIDE;
  const int cnt = fl[0];
  if (cnt == 0 || cnt > GR_CAP) return;
  const Img im = imgs[blockIdx.z];
  const long plane = (long)im.h * im.w;
  double *E = energy[blockIdx.z] + f * plane;
  float *D = bound[blockIdx.z] + f * plane;
  const gptr<const double> K = to_global(kernels + (long)f * GB_N * GB_N * 2);
  const gptr<const double> px = to_global((const double *)im.p);
  const int lane = threadIdx.x;
  for (int k = 0; k < cnt; k++) {
    const int i = fl[1 + k];
    const int y = i / im.w, x = i - y * im.w;
    for (int tp = lane; tp < GB_N * GB_N; tp += 64) {
      const int j = tp / GB_N, c = tp - j * GB_N;
      const int yy = y + 19 - j, xx = x + 19 - c;
      const double v = (yy >= 0 && yy < im.h && xx >= 0 && xx < im.w) ? px[(long)yy * im.w + xx] : 0.0;
      pre[tp] = v * K[2 * tp];
      pim[tp] = v * K[2 * tp + 1];
    }
    __syncthreads();
    if (lane == 0) {
      double re = 0.0, imv = 0.0;
      int tp = 0;
      for (; tp + 8 <= GB_N * GB_N; tp += 8) {  // eight products read at a time, added in order
        double a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          a[u] = pre[tp + u];
          b[u] = pim[tp + u];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
          re += a[u];
          imv += b[u];
        }
      }
      for (; tp < GB_N * GB_N; tp++) {
        re += pre[tp];
        imv += pim[tp];
      }
      E[i] = sqrt(re * re + imv * imv);
      D[i] = 0.0f;
    }
    __syncthreads();  // the products of the next energy overwrite these
  }
}

__global__ void __launch_bounds__(256) k_gabor_repair(const Img *imgs, const double *kernels, double *const *energy,
                                                      float *const *bound, const int *flags, int loop_tiles) {
  __shared__ double tile[GB_TR + GB_N - 1][GB_LD];
  __shared__ double2 wk[GB_N * GB_N];
  __shared__ int list[GB_TR * GB_TC];
  __shared__ int nlist;
  const int f = blockIdx.y;
  if (flags[(long)(blockIdx.z * 8 + f) * GR_STRIDE] <= GR_CAP) return;  // none, or listed
  const Img im = imgs[blockIdx.z];
  const int ntiles = ((im.w + GB_TC - 1) / GB_TC) * ((im.h + GB_TR - 1) / GB_TR);
  const long plane = (long)im.h * im.w;
  double *E = energy[blockIdx.z] + f * plane;
  float *D = bound[blockIdx.z] + f * plane;
  const double *K = kernels + (long)f * GB_N * GB_N * 2;
  if (loop_tiles) {
    for (int tl = 0; tl < ntiles; tl++) gabor_repair_tile(im, tl, K, E, D, tile, wk, list, &nlist);
  } else if ((int)blockIdx.x < ntiles) {
    gabor_repair_tile(im, blockIdx.x, K, E, D, tile, wk, list, &nlist);
  }
}

// What the phases of the post-processing pass on, per (image, filter); values
// that are minima or maxima over blocks are kept by their order-preserving keys.
// GaborState is declared in kernels.hpp, for the caller's scratch.
//
// A phase first forms what it needs over the plane and then marks: two steps
// (phase 2 three, filter 0 going straight on), each over blocks of GP_CHUNK
// pixels.  Bound by memory: 12 bytes per pixel and filter and step.  Three planes
// of 1388 x 1040: 0.8 ms for all steps, 10.1 ms with one block per (image,
// filter); 64 planes of 64..1024 pixels a side: 2.6, 8.1 ms; 400 of 256 x 256:
// 4.3, 4.5 ms; one of 128 x 128: 0.115, 0.12 ms (the threshold's chain of 1,024
// bins and the launches).
enum GaborStep { GP_LOW, GP_MARK_TOP, GP_MAX, GP_LEVEL, GP_MARK_LOW, GP_RANGE, GP_MARK_BIN, GP_HIST, GP_MARK_THR, GP_COUNT };
constexpr int GP_CHUNK = 8192;

__global__ void __launch_bounds__(1024) k_gabor_init(GaborState *state, int *flags, int count) {
  for (int e = blockIdx.x; e < count; e += gridDim.x) {
    GaborState &S = state[e];
    S.hist[threadIdx.x] = 0;
    if (threadIdx.x == 0) {
      S.lo = S.mx = S.b = dkey(-1e308);
      S.hi_min = S.a = dkey(1e308);
      S.base = S.above = 0;
      flags[(long)e * GR_STRIDE] = 0;
    }
  }
}

template <int STEP>
__global__ void __launch_bounds__(256) k_gabor_step(const Img *imgs, double *const *energy, float *const *bound,
                                                    GaborState *state, int *flags) {
  __shared__ int hist[STEP == GP_HIST ? 1024 : 1];
  __shared__ double shd[4];
  __shared__ int shi[4];
  constexpr bool MARKS = STEP == GP_MARK_TOP || STEP == GP_LEVEL || STEP == GP_MARK_LOW || STEP == GP_MARK_BIN || STEP == GP_MARK_THR;
  const Img im = imgs[blockIdx.z];
  const long n = (long)im.h * im.w, c0 = (long)blockIdx.x * GP_CHUNK;
  if (c0 >= n) return;
  const int f = blockIdx.y, e = blockIdx.z * 8 + f;
  GaborState &S = state[e];
  int *fl = flags + (long)e * GR_STRIDE;
  // the marks of the last phase are repaired; the next ones come in a later step
  if ((STEP == GP_MAX || STEP == GP_RANGE || STEP == GP_HIST) && c0 == 0 && threadIdx.x == 0) fl[0] = 0;
  if ((STEP == GP_MARK_LOW || STEP == GP_MARK_BIN || STEP == GP_HIST || STEP == GP_MARK_THR || STEP == GP_COUNT) && f == 0) return;
  const gptr<const double> E = to_global((const double *)(energy[blockIdx.z] + f * n));
  float *const Dp = bound[blockIdx.z] + f * n;
  const gptr<const float> Dg = to_global((const float *)Dp);
  const double mx = STEP >= GP_LEVEL ? dkey_inv(S.mx) : 0.0;
  const double lo = STEP == GP_MARK_TOP ? dkey_inv(S.lo) : 0.0, hi_min = STEP == GP_MARK_LOW ? dkey_inv(S.hi_min) : 0.0;
  const double a = STEP >= GP_MARK_BIN ? dkey_inv(S.a) : 0.0, b = STEP >= GP_MARK_BIN ? dkey_inv(S.b) : 0.0;
  const double thr = STEP >= GP_MARK_THR ? S.thr : 0.0;
  const double sc = STEP == GP_MARK_BIN || STEP == GP_HIST ? hist_scale(a, b, 1024) : 0.0;
  if (STEP == GP_MARK_LOW && !(mx > 0)) return;
  if (STEP == GP_HIST) {
    for (int k = threadIdx.x; k < 1024; k += 256) hist[k] = 0;
    __syncthreads();
  }
  double vmax = -1e308, vmin = 1e308;
  int cnt = 0;
  const long end = min(n, c0 + GP_CHUNK);
  for (long i0 = c0 + threadIdx.x; i0 < end; i0 += 256 * 4) {
    double ev[4];
    float dv[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const long i = min(i0 + 256 * k, end - 1);
      ev[k] = E[i];
      dv[k] = Dg[i];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const long i = i0 + 256 * k;
      if (i >= end) continue;
      const double x = ev[k], d = dv[k];
      const bool exact = dv[k] == 0.0f;
      bool mark = false;
      if (STEP == GP_LOW) vmax = fmax(vmax, x - d);
      if (STEP == GP_MARK_TOP) mark = !exact && x + d >= lo;
      if (STEP == GP_MAX && exact) vmax = fmax(vmax, x);  // nothing else can reach the candidates
      if (STEP == GP_LEVEL) {
        if (!(mx > 0)) mark = !exact;  // no energy: every value exact, then the FP64 rules as written
        else if (f == 0) mark = !exact && x - d <= mx * 0.4 && x + d > mx * 0.4;
        else {
          const double v = (x + d) / mx;
          if (moments_ok(v)) vmin = fmin(vmin, v);
        }
      }
      if (STEP == GP_MARK_LOW) mark = !exact && (x - d) / mx <= hi_min;
      if (STEP == GP_RANGE) {
        if (f == 0) cnt += exact ? x > mx * 0.4 : x - d > mx * 0.4;  // open pixels were recomputed
        else {
          const double v = x / mx;
          if (exact && moments_ok(v)) { vmin = fmin(vmin, v); vmax = fmax(vmax, v); }
        }
      }
      if (STEP == GP_MARK_BIN && !exact) {
        // the true value lies in [a, b]: clamp the interval's ends there
        const double vl = fmax((x - d) / mx, a), vh = fmin((x + d) / mx, b);
        mark = hist_bin(vl, a, sc, 1024) != hist_bin(vh, a, sc, 1024);
      }
      if (STEP == GP_HIST) {
        // d > 0: the bin was decided by the interval (both ends give it)
        const double v = exact ? x / mx : fmax((x - d) / mx, a);
        atomicAdd(&hist[hist_bin(v, a, sc, 1024)], 1);
      }
      if (STEP == GP_MARK_THR) mark = !exact && (x - d) / mx <= thr && (x + d) / mx > thr;
      if (STEP == GP_COUNT) cnt += exact ? (x / mx) > thr : (x - d) / mx > thr;
      if (MARKS && mark) {
        Dp[i] = -dv[k];
        const int q = atomicAdd(fl, 1);
        if (q < GR_CAP) fl[1 + q] = (int)i;
      }
    }
  }
  if (STEP == GP_LOW || STEP == GP_MAX || STEP == GP_RANGE) vmax = block_reduce(vmax, MaxOp(), shd);
  if (STEP == GP_LEVEL || STEP == GP_RANGE) vmin = block_reduce(vmin, MinOp(), shd);
  if (STEP == GP_RANGE || STEP == GP_COUNT) cnt = block_reduce(cnt, SumOp(), shi);
  if (threadIdx.x == 0) {
    if (STEP == GP_LOW) atomicMax(&S.lo, (unsigned long long)dkey(vmax));
    if (STEP == GP_MAX) atomicMax(&S.mx, (unsigned long long)dkey(vmax));
    if (STEP == GP_LEVEL) atomicMin(&S.hi_min, (unsigned long long)dkey(vmin));
    if (STEP == GP_RANGE) {
      atomicMin(&S.a, (unsigned long long)dkey(vmin));
      atomicMax(&S.b, (unsigned long long)dkey(vmax));
      if (f == 0) atomicAdd(&S.base, (unsigned long long)cnt);
    }
    if (STEP == GP_COUNT) atomicAdd(&S.above, (unsigned long long)cnt);
  }
  if (STEP == GP_HIST) {
    __syncthreads();
    for (int k = threadIdx.x; k < 1024; k += 256)
      if (hist[k]) atomicAdd(&S.hist[k], hist[k]);
  }
}

__global__ void __launch_bounds__(1024) k_gabor_threshold(const Img *imgs, GaborState *state) {
  __shared__ int hist[1024];
  const Img im = imgs[blockIdx.x];
  GaborState &S = state[blockIdx.x * 8 + blockIdx.y + 1];
  hist[threadIdx.x] = S.hist[threadIdx.x];
  __syncthreads();
  const double thr = otsu_threshold(hist, (long)im.h * im.w, dkey_inv(S.a), dkey_inv(S.b));
  if (threadIdx.x == 0) S.thr = thr;
}

__global__ void __launch_bounds__(64) k_gabor_ratios(const GaborState *state, OutRef o) {
  const int f = threadIdx.x;
  if (f >= 1 && f < 8)
    o.rows[blockIdx.x][f - 1] = (double)state[blockIdx.x * 8 + f].above / (double)state[blockIdx.x * 8].base;
}

void launch_gabor_post_exact(const Img *imgs, double *const *energy, float *const *bound, const double *taps,
                             GaborState *state, int *flags, bool loop_tiles, OutRef o, int nimg, int maxh, int maxw,
                             hipStream_t s) {
  const int tiles = loop_tiles ? 1 : ((maxw + GB_TC - 1) / GB_TC) * ((maxh + GB_TR - 1) / GB_TR);
  const dim3 grid((unsigned)(((long)maxh * maxw + GP_CHUNK - 1) / GP_CHUNK), 8, nimg);
  auto repair = [&] {
    k_gabor_repair_list<<<dim3(1, 8, nimg), 64, 0, s>>>(imgs, taps, energy, bound, flags);
    k_gabor_repair<<<dim3(tiles, 8, nimg), 256, 0, s>>>(imgs, taps, energy, bound, flags, loop_tiles);
  };
  k_gabor_init<<<std::min(8 * nimg, 4096), 1024, 0, s>>>(state, flags, 8 * nimg);
  k_gabor_step<GP_LOW><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  k_gabor_step<GP_MARK_TOP><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  repair();
  k_gabor_step<GP_MAX><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  k_gabor_step<GP_LEVEL><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  k_gabor_step<GP_MARK_LOW><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  repair();
  k_gabor_step<GP_RANGE><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  k_gabor_step<GP_MARK_BIN><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  repair();
  k_gabor_step<GP_HIST><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  k_gabor_threshold<<<dim3(nimg, 7), 1024, 0, s>>>(imgs, state);
  k_gabor_step<GP_MARK_THR><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  repair();
  k_gabor_step<GP_COUNT><<<grid, 256, 0, s>>>(imgs, energy, bound, state, flags);
  k_gabor_ratios<<<nimg, 64, 0, s>>>(state, o);
}

void launch_gabor(const Img *imgs, const double *kernels, double *const *energy, OutRef o, int nimg, int maxh,
                  int maxw, hipStream_t s) {
  const int tiles = ((maxw + GB_TC - 1) / GB_TC) * ((maxh + GB_TR - 1) / GB_TR);
  k_gabor_conv<<<dim3(tiles, 8, nimg), 256, 0, s>>>(imgs, kernels, energy);
  k_gabor_post<<<nimg, 1024, 0, s>>>(imgs, energy, o);
}
void launch_gabor_certified(const Img *imgs, const double *kernels, const double *factors, const double *wsum,
                            double slack, double *const *energy, float *const *bound, GaborState *state, int *flags,
                            OutRef o, int nimg, int maxh, int maxw, hipStream_t s) {
  const int tiles = ((maxw + GB_TC - 1) / GB_TC) * ((maxh + GS_TR - 1) / GS_TR);
  // a CU holds one block: from two blocks per CU on, the input tile is read once
  // for all filters, below that the filters go to blocks of their own (one image
  // of 128 x 128: 10 blocks or 80)
  const int per = (long)tiles * nimg >= 512 ? 8 : 1;
  k_gabor_sep<<<dim3(tiles, 8 / per, nimg), 512, 0, s>>>(imgs, factors, kernels, energy, wsum, bound, 4e-13 * slack, per);
  launch_gabor_post_exact(imgs, energy, bound, kernels, state, flags, slack <= 1.0, o, nimg, maxh, maxw, s);
}

}  // namespace wnd
