// Lanczos vector kernels, tridiagonal eigensolver and the device generator.
#include "lanczos.hpp"
#include "wave.hpp"

#include <algorithm>
#include <cfloat>
#include <cmath>

namespace dmrg {
namespace {

// The vector kernels run 1024 threads on chunks of 1024 E elements, thread t of
// workgroup b on the elements b 1024 E + 1024 e + t, held in registers: one
// workgroup a CU up to 2^20 elements, so the partial sums that the next kernel
// reduces stay at 256 a value.
constexpr int NT = 256;
constexpr int NL = 1024;
constexpr int NW = NL / 64;

template <class T> struct Acc;
template <> struct Acc<double> {
  static constexpr int N = 1;
  __device__ static void put(double v, double* o) { o[0] = v; }
  __device__ static double get(const double* o) { return o[0]; }
};
template <> struct Acc<cdouble> {
  static constexpr int N = 2;
  __device__ static void put(cdouble v, double* o) { o[0] = v.x; o[1] = v.y; }
  __device__ static cdouble get(const double* o) { return cdouble(o[0], o[1]); }
};

// Reductions across workgroups carry no fence or atomic: each producing
// kernel writes one partial per workgroup, and the kernel that consumes the
// sum re-reduces the partials itself (every wave, same fixed order, so all see
// bit-identical values).  The kernel boundary makes the partials visible.  A
// device-scope release inside a kernel would write back the L2 of every XCD
// once per wave.

// Sum of part[0..nb) in every lane of the calling wave.
__device__ inline double sum_parts(const double* __restrict__ part, int nb) {
  double s = 0.0;
  for (int b = threadIdx.x & 63; b < nb; b += 64) s += part[b];
  return wave_sum_all(s);
}

// A sum that the consuming kernel forms with sum_parts: n partials at p.
struct Parts {
  const double* p;
  int n;
};

// Sum of v over the workgroup, in every thread (sh: NW values, free on return).
__device__ inline double block_sum(double v, double* sh) {
  v = wave_sum_all(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < NW; ++i) r += sh[i];
  __syncthreads();
  return r;
}

// The thread's elements of x (zero, and an index inside the vector, past n):
// base + off[e], the base uniform over the workgroup.
template <int E>
struct Chunk {
  size_t base;
  unsigned off[E];
  bool in[E];
  __device__ explicit Chunk(size_t n) : base((size_t)blockIdx.x * (E * NL)) {
    const size_t left = n - base;  // at least one element for every workgroup
    const unsigned cnt = left < E * NL ? (unsigned)left : E * NL;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const unsigned i = e * NL + threadIdx.x;
      in[e] = i < cnt;
      off[e] = in[e] ? i : cnt - 1;
    }
  }
  template <class T> __device__ void load(const T* __restrict__ x, T (&v)[E]) const {
    x += base;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const T u = x[off[e]];
      v[e] = in[e] ? u : T(0);
    }
  }
  template <class T> __device__ void store(T* __restrict__ x, const T (&v)[E]) const {
    x += base;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (in[e]) x[off[e]] = v[e];
  }
};
template <class T, int E> __device__ inline double sum_abs2(const T (&v)[E]) {
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) s += abs2(v[e]);
  return s;
}

// Basis vectors taken at once: their loads are in flight together.
template <class T, int E> constexpr int group() {
  return E == 1 ? 8 : (is_cplx<T>::value ? 8 : 16) / E;
}
// v[g] = the thread's elements of basis vector j0 + g (of the last one past cnt).
template <class T, int E, int G>
__device__ inline void load_group(const Chunk<E>& c, const T* __restrict__ V, size_t n, int j0,
                                  int cnt, T (&v)[G][E]) {
#pragma unroll
  for (int g = 0; g < G; ++g) c.load(V + (size_t)min(j0 + g, cnt - 1) * n, v[g]);
}

// sh[(j NC + c) NW + wave] = the wave's part of <v_j, x>, j < cnt.  v holds
// the first group.
template <class T, int E, int G>
__device__ inline void wave_dots(const Chunk<E>& c, const T* __restrict__ V, size_t n, int cnt,
                                 const T (&x)[E], T (&v)[G][E], double* sh) {
  constexpr int NC = Acc<T>::N;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int j0 = 0; j0 < cnt; j0 += G) {
    if (j0 > 0) load_group<T, E, G>(c, V, n, j0, cnt, v);
    double o[G * NC];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      T a = conj(v[g][0]) * x[0];
#pragma unroll
      for (int e = 1; e < E; ++e) a += conj(v[g][e]) * x[e];
      Acc<T>::put(a, o + g * NC);
    }
#pragma unroll
    for (int q = 0; q < G * NC; ++q) o[q] = wave_sum_all(o[q]);
    if (lane == 0)
#pragma unroll
      for (int q = 0; q < G * NC; ++q)
        if (j0 * NC + q < cnt * NC) sh[(j0 * NC + q) * NW + w] = o[q];
  }
}

// x -= sum_j c_j v_j, j < cnt.  v holds the first group.
template <class T, int E, int G>
__device__ inline void sub_basis(const Chunk<E>& c, const T* __restrict__ V, size_t n, int cnt,
                                 const double* cs, T (&x)[E], T (&v)[G][E]) {
  constexpr int NC = Acc<T>::N;
  for (int j0 = 0; j0 < cnt; j0 += G) {
    if (j0 > 0) load_group<T, E, G>(c, V, n, j0, cnt, v);
#pragma unroll
    for (int g = 0; g < G; ++g)
      if (j0 + g < cnt) {
        const T cj = Acc<T>::get(cs + (j0 + g) * NC);
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] -= cj * v[g][e];
      }
  }
}

// partN[blk] = sum |x_i|^2 over the chunk; starts a Lanczos call.
template <class T, int E>
__global__ __launch_bounds__(NL) void k_norm(const T* __restrict__ x, size_t n,
                                            double* __restrict__ partN, double* scal) {
  __shared__ double sh[NW];
  const Chunk<E> c(n);
  T v[E];
  c.load(x, v);
  const double s = block_sum(sum_abs2<T, E>(v), sh);
  if (threadIdx.x == 0) partN[blockIdx.x] = s;
  if (blockIdx.x == 0 && threadIdx.x == 0) scal[2] = 1e30;
}

__device__ inline double u_pm1(uint64_t seed, uint64_t k) {
  uint64_t z = seed + (k + 1ull) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return 2.0 * ((double)(z >> 11) * (1.0 / 9007199254740992.0)) - 1.0;
}
template <class T> __device__ inline T rand_entry(uint64_t seed, uint64_t idx, double scale);
template <> __device__ inline double rand_entry<double>(uint64_t seed, uint64_t idx, double scale) {
  return u_pm1(seed, idx) * scale;
}
template <> __device__ inline cdouble rand_entry<cdouble>(uint64_t seed, uint64_t idx, double scale) {
  return cdouble(u_pm1(seed, 2 * idx) * scale, u_pm1(seed, 2 * idx + 1) * scale);
}

// Fill x from the stream.
template <class T>
__global__ __launch_bounds__(NT) void k_fill_random(T* x, size_t n, uint64_t seed, uint64_t offset,
                                                   double scale) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    x[i] = rand_entry<T>(seed, offset + i, scale);
}

// x <- the stream when sqrt(sum partN) < thr; partO: the norm partials of the
// result.
template <class T, int E>
__global__ __launch_bounds__(NL) void k_fill_small(T* x, size_t n, uint64_t seed, double thr,
                                                  const double* __restrict__ partN, Parts sumN,
                                                  double* __restrict__ partO) {
  __shared__ double sh[NW];
  if (!(sqrt(sum_parts(sumN.p, sumN.n)) < thr)) {
    if (threadIdx.x == 0) partO[blockIdx.x] = partN[blockIdx.x];
    return;
  }
  const Chunk<E> c(n);
  T v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = c.in[e] ? rand_entry<T>(seed, c.base + c.off[e], 1.0) : T(0);
  c.store(x, v);
  const double s = block_sum(sum_abs2<T, E>(v), sh);
  if (threadIdx.x == 0) partO[blockIdx.x] = s;
}

// scal[0] = nrm, scal[1] = s, *beta = nrm; host[0] = nrm, host[3] = scal[3] (each if given)
__device__ inline void put_norm(double nrm, double s, double* scal, double* beta, double* host) {
  scal[0] = nrm;
  scal[1] = s;
  if (beta) *beta = nrm;
  if (host) {
    host[0] = nrm;
    host[3] = scal[3];
  }
}
__device__ inline double inv_norm(double nrm) { return (nrm > 1e-300) ? 1.0 / nrm : 0.0; }

// nrm = sqrt(sum partN); dst = src / nrm (if dst given; zero if nrm <= 1e-300).
template <class T, int E>
__global__ __launch_bounds__(NL) void k_scale(T* dst, const T* src, size_t n,
                                             Parts sumN, double* scal, double* beta_out,
                                             double* host) {
  const Chunk<E> c(n);
  T v[E];
  c.load(src, v);
  const double nrm = sqrt(sum_parts(sumN.p, sumN.n));
  const double s = inv_norm(nrm);
  if (blockIdx.x == 0 && threadIdx.x == 0) put_norm(nrm, s, scal, beta_out, host);
  if (!dst) return;
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = v[e] * s;
  c.store(dst, v);
}

// partA[blk] = Re <v, w> over the chunk.
template <class T, int E>
__global__ __launch_bounds__(NL) void k_alpha(const T* __restrict__ v, const T* __restrict__ w,
                                             size_t n, double* __restrict__ partA) {
  __shared__ double sh[NW];
  const Chunk<E> c(n);
  T a[E], b[E];
  c.load(v, a);
  c.load(w, b);
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) s += real(conj(a[e]) * b[e]);
  s = block_sum(s, sh);
  if (threadIdx.x == 0) partA[blockIdx.x] = s;
}

// alpha[it] = sum partA;  w -= alpha v_it + beta[it-1] v_{it-1};
// partC[(j*NC + c)*nb + blk] = component c of <v_j, w> over the chunk, j <= it.
// One pass over the basis, bound by the L2 and the Infinity Cache; every load
// of a group of vectors is in flight before the first sum is needed (n = 2^18,
// 20 iterations: 17.6 -> 8.3 us on average; four waves a CU and a reduction
// through LDS per group of eight vectors before).
template <class T, int E>
__global__ __launch_bounds__(NL) void k_sub_dots(T* __restrict__ w, const T* __restrict__ V,
                                                size_t n, int it, Parts sumA, double* alpha,
                                                const double* beta,
                                                double* __restrict__ partC) {
  constexpr int NC = Acc<T>::N, G = group<T, E>();
  __shared__ double sh[128 * NC * NW];
  const int nb = gridDim.x, cnt = it + 1;
  const Chunk<E> c(n);
  T x[E], vi[E], vm[E], v[G][E];
  c.load(w, x);
  c.load(V + (size_t)it * n, vi);
  c.load(V + (size_t)max(it - 1, 0) * n, vm);
  load_group<T, E, G>(c, V, n, 0, cnt, v);
  const double a = sum_parts(sumA.p, sumA.n);
  const double bm = it > 0 ? beta[it - 1] : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) alpha[it] = a;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    x[e] = x[e] - a * vi[e];
    if (it > 0) x[e] = x[e] - bm * vm[e];
  }
  c.store(w, x);
  wave_dots<T, E, G>(c, V, n, cnt, x, v, sh);
  __syncthreads();
  for (int q = threadIdx.x; q < cnt * NC; q += NL) {
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < NW; ++i) r += sh[q * NW + i];
    partC[(size_t)q * nb + blockIdx.x] = r;
  }
}

// out[g] = sum_b part[g*nb + b] (one workgroup of NTH threads per g, fixed order).
template <int NTH>
__global__ __launch_bounds__(NTH) void k_totals(const double* __restrict__ part, int nb,
                                                double* __restrict__ out) {
  const double* const p = part + (size_t)blockIdx.x * nb;
  double s;
  if constexpr (NTH == 64) {
    s = sum_parts(p, nb);
  } else {
    __shared__ double sh[NW];
    s = 0.0;
    for (int b = threadIdx.x; b < nb; b += NTH) s += p[b];
    s = block_sum(s, sh);
  }
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// w -= sum_j c_j v_j (c from cvec, or re-reduced from partC when cvec is null);
// partN[blk] = |w|^2 over the chunk.
template <class T, int E>
__global__ __launch_bounds__(NL) void k_orth_norm(T* __restrict__ w, const T* __restrict__ V,
                                                 size_t n, int it, const double* __restrict__ partC,
                                                 const double* __restrict__ cvec,
                                                 double* __restrict__ partN) {
  constexpr int NC = Acc<T>::N, G = group<T, E>();
  __shared__ double sh[NW];
  __shared__ double cs[128 * NC];
  const int nb = gridDim.x, cnt = it + 1;
  const Chunk<E> c(n);
  T x[E], v[G][E];
  c.load(w, x);
  load_group<T, E, G>(c, V, n, 0, cnt, v);
  if (cvec) {
    for (int q = threadIdx.x; q < cnt * NC; q += NL) cs[q] = cvec[q];
  } else {
    for (int q = threadIdx.x >> 6; q < cnt * NC; q += NW) {
      const double r = sum_parts(partC + (size_t)q * nb, nb);
      if ((threadIdx.x & 63) == 0) cs[q] = r;
    }
  }
  __syncthreads();
  sub_basis<T, E, G>(c, V, n, cnt, cs, x, v);
  c.store(w, x);
  const double s = block_sum(sum_abs2<T, E>(x), sh);
  if (threadIdx.x == 0) partN[blockIdx.x] = s;
}

// out = sum_j y_j v_j; partN[blk] = |out|^2 over the chunk.
template <class T, int E>
__device__ inline double ritz_chunk(const Chunk<E>& c, const T* __restrict__ V, size_t n, int niter,
                                    const double* ys, T (&x)[E]) {
  constexpr int G = group<T, E>();
#pragma unroll
  for (int e = 0; e < E; ++e) x[e] = T(0);
  for (int j0 = 0; j0 < niter; j0 += G) {
    T v[G][E];
    load_group<T, E, G>(c, V, n, j0, niter, v);
#pragma unroll
    for (int g = 0; g < G; ++g)
      if (j0 + g < niter)
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] += ys[j0 + g] * v[g][e];
  }
  return sum_abs2<T, E>(x);
}
template <class T, int E>
__global__ __launch_bounds__(NL) void k_ritz(T* __restrict__ out, const T* __restrict__ V, size_t n,
                                            int niter, const double* y, double* __restrict__ partN) {
  __shared__ double sh[NW];
  __shared__ double ys[128];
  for (int j = threadIdx.x; j < niter; j += NL) ys[j] = y[j];
  __syncthreads();
  const Chunk<E> c(n);
  T x[E];
  const double s = block_sum(ritz_chunk<T, E>(c, V, n, niter, ys, x), sh);
  c.store(out, x);
  if (threadIdx.x == 0) partN[blockIdx.x] = s;
}

// ---------------------------------------------------------------------------
// Vectors of at most LZ_ONE elements: one workgroup holds the vector, so an
// iteration's four kernels (and the three at either end of a call) are one.
// Such launches cost their latency, not their work (20 iterations with the
// two-site operator, one workgroup against four kernels: n = 256 473 us against
// 676, 1024 500 against 688).  Past LZ_ONE the basis through one CU takes what
// the launches save (n = 2304 717 against 721, 6400 1138 against 782).
// ---------------------------------------------------------------------------
// v_0 = theta / |theta|, theta replaced by the stream when |theta| < thr.
template <class T, int E>
__global__ __launch_bounds__(NL) void k_one_start(T* theta, T* v0, size_t n, uint64_t seed,
                                                 double thr, double* scal) {
  __shared__ double sh[NW];
  const Chunk<E> c(n);
  T x[E];
  c.load(theta, x);
  double nrm = sqrt(block_sum(sum_abs2<T, E>(x), sh));
  if (nrm < thr) {
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = c.in[e] ? rand_entry<T>(seed, c.base + c.off[e], 1.0) : T(0);
    c.store(theta, x);
    nrm = sqrt(block_sum(sum_abs2<T, E>(x), sh));
  }
  const double s = inv_norm(nrm);
  if (threadIdx.x == 0) {
    put_norm(nrm, s, scal, nullptr, nullptr);
    scal[2] = 1e30;
  }
#pragma unroll
  for (int e = 0; e < E; ++e) x[e] = x[e] * s;
  c.store(v0, x);
}

// One iteration behind w = H v_it: alpha[it], the three-term update, one
// projection on the basis, beta[it] and v_{it+1} (if given).
template <class T, int E>
__global__ __launch_bounds__(NL) void k_one_step(const T* __restrict__ w, T* V, size_t n, int it,
                                                double* alpha, double* beta, double* scal,
                                                T* vnext) {
  constexpr int NC = Acc<T>::N, G = group<T, E>();
  __shared__ double sh[128 * NC * NW];
  __shared__ double cs[128 * NC];
  const int cnt = it + 1;
  const Chunk<E> c(n);
  T x[E], vi[E], vm[E], v[G][E];
  c.load(w, x);
  c.load(V + (size_t)it * n, vi);
  c.load(V + (size_t)max(it - 1, 0) * n, vm);
  load_group<T, E, G>(c, V, n, 0, cnt, v);
  const double bm = it > 0 ? beta[it - 1] : 0.0;
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) s += real(conj(vi[e]) * x[e]);
  const double a = block_sum(s, sh);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    x[e] = x[e] - a * vi[e];
    if (it > 0) x[e] = x[e] - bm * vm[e];
  }
  wave_dots<T, E, G>(c, V, n, cnt, x, v, sh);
  load_group<T, E, G>(c, V, n, 0, cnt, v);
  __syncthreads();
  for (int q = threadIdx.x; q < cnt * NC; q += NL) {
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < NW; ++i) r += sh[q * NW + i];
    cs[q] = r;
  }
  __syncthreads();
  sub_basis<T, E, G>(c, V, n, cnt, cs, x, v);
  const double nrm = sqrt(block_sum(sum_abs2<T, E>(x), sh));
  const double si = inv_norm(nrm);
  if (threadIdx.x == 0) {
    alpha[it] = a;
    put_norm(nrm, si, scal, beta + it, nullptr);
  }
  if (!vnext) return;
#pragma unroll
  for (int e = 0; e < E; ++e) x[e] = x[e] * si;
  c.store(vnext, x);
}

// out = V y / |V y|
template <class T, int E>
__global__ __launch_bounds__(NL) void k_one_ritz(T* __restrict__ out, const T* __restrict__ V,
                                                size_t n, int niter, const double* y, double* scal,
                                                double* host) {
  __shared__ double sh[NW];
  __shared__ double ys[128];
  for (int j = threadIdx.x; j < niter; j += NL) ys[j] = y[j];
  __syncthreads();
  const Chunk<E> c(n);
  T x[E];
  const double nrm = sqrt(block_sum(ritz_chunk<T, E>(c, V, n, niter, ys, x), sh));
  const double s = inv_norm(nrm);
  if (threadIdx.x == 0) put_norm(nrm, s, scal, nullptr, host);
#pragma unroll
  for (int e = 0; e < E; ++e) x[e] = x[e] * s;
  c.store(out, x);
}

// ---------------------------------------------------------------------------
// Symmetric tridiagonal T(k): diagonal a[0..k), off-diagonal b[0..k-1).
// ---------------------------------------------------------------------------

// Lowest eigenvalue by multisection (one wave): every lane holds the same
// bracket [lo, hi] (the same arithmetic on the same data) and tests two of 128
// interior points a round; ballots give the first point x at which T - x I is
// not positive definite.  The test is the sign of the leading minors,
// p_{i+1} = (a_i - x) p_i - b_{i-1}^2 p_{i-1}: one multiply-add of latency a
// row where the recurrence of their ratios has a division, and as the ratios
// exact for a matrix an eps away.  T is scaled by a power of two to entries
// below 4 and the pair of minors every eight rows, so neither leaves the range.
// A check of 7 to 19 rows takes 7 to 10 us (12 to 16 with divisions).
__device__ double tri_lowest(const double* a, const double* b, int k, double* as /*[144]*/,
                             double* b2 /*[144]*/) {
  const int t = threadIdx.x;
  double lo = INFINITY, hi = -INFINITY, bad = 0.0;
  for (int i = t; i < k; i += 64) {
    const double r = (i > 0 ? fabs(b[i - 1]) : 0.0) + (i < k - 1 ? fabs(b[i]) : 0.0);
    lo = fmin(lo, a[i] - r);
    hi = fmax(hi, a[i] + r);
    bad += 0.0 * a[i] + 0.0 * r;  // NaN for an infinite or NaN entry
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o, 64));
    hi = fmax(hi, __shfl_xor(hi, o, 64));
    bad += __shfl_xor(bad, o, 64);
  }
  if (!(bad == 0.0) || !(hi - lo < INFINITY)) return NAN;
  const double w0 = fmax(fabs(lo), fabs(hi));
  lo -= 2.0 * DBL_EPSILON * w0 + DBL_MIN;
  hi += 2.0 * DBL_EPSILON * w0 + DBL_MIN;
  const int ex = ilogb(fmax(w0, 1e-290));
  // rows past k: a = 8 and b = 0 keep the sign of the minors
  for (int i = t; i < 144; i += 64) {
    as[i] = i < k ? ldexp(a[min(i, k - 1)], -ex) : 8.0;
    const double bi = i > 0 && i < k ? ldexp(b[min(i, k - 1) - (i > 0)], -ex) : 0.0;
    b2[i] = bi * bi;
  }
  __syncthreads();
  lo = ldexp(lo, -ex);
  hi = ldexp(hi, -ex);
  for (int round = 0; round < 20; ++round) {
    const double w = fmax(fabs(lo), fabs(hi));
    if (hi - lo <= 2.0 * DBL_EPSILON * w + 4.0 * DBL_MIN) break;
    const double x0 = lo + (hi - lo) * (double)(t + 1) / 129.0;
    const double x1 = lo + (hi - lo) * (double)(t + 65) / 129.0;
    double p0 = 1.0, q0 = 0.0, p1 = 1.0, q1 = 0.0;
    bool n0 = false, n1 = false;
    double ca[8], cb[8];  // the next eight rows, read ahead of the chain
#pragma unroll
    for (int u = 0; u < 8; ++u) ca[u] = as[u], cb[u] = b2[u];
    for (int i0 = 0; i0 < k; i0 += 8) {
      double ra[8], rb[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        ra[u] = ca[u], rb[u] = cb[u];
        ca[u] = as[i0 + 8 + u], cb[u] = b2[i0 + 8 + u];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const double r0 = (ra[u] - x0) * p0 - rb[u] * q0, r1 = (ra[u] - x1) * p1 - rb[u] * q1;
        q0 = p0, p0 = r0;
        q1 = p1, p1 = r1;
        n0 |= !(r0 > 0.0);
        n1 |= !(r1 > 0.0);
      }
      const int e0 = __builtin_amdgcn_frexp_exp(fmax(fabs(p0), fabs(q0)));
      const int e1 = __builtin_amdgcn_frexp_exp(fmax(fabs(p1), fabs(q1)));
      p0 = ldexp(p0, -e0), q0 = ldexp(q0, -e0);
      p1 = ldexp(p1, -e1), q1 = ldexp(q1, -e1);
    }
    const unsigned long long m0 = __ballot(n0), m1 = __ballot(n1);
    const int l = m0 ? __ffsll((long long)m0) - 1 : m1 ? 63 + __ffsll((long long)m1) : 128;
    const double nlo = (l == 0) ? lo : lo + (hi - lo) * (double)l / 129.0;
    const double nhi = (l == 128) ? hi : lo + (hi - lo) * (double)(l + 1) / 129.0;
    lo = nlo;
    hi = nhi;
  }
  return ldexp(0.5 * (lo + hi), ex);
}

// Eigenvector of T for eigenvalue lam by inverse iteration (one wave): thread 0
// factors T - lam I with partial pivoting and runs the two substitutions; the
// wave inverts the pivots and normalises.  Work arrays in LDS.
struct TriWork {
  double d[128], du[128], dl[128], du2[128], x[128];
  int piv[128];
};
__device__ inline double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ void tri_vector(const double* a, const double* b, int k, double lam, double* y,
                           TriWork& s) {
  const int t = threadIdx.x;
  double tnorm = 0.0;
  for (int i = t; i < k; i += 64) {
    tnorm = fmax(tnorm, fabs(a[i]) + (i > 0 ? fabs(b[i - 1]) : 0.0) + (i < k - 1 ? fabs(b[i]) : 0.0));
    s.d[i] = a[i] - lam;
    s.du[i] = s.dl[i] = i < k - 1 ? b[i] : 0.0;
    s.du2[i] = 0.0;
    s.x[i] = 1.0 + 0.25 * (double)i / (double)k;
  }
  tnorm = wave_max(tnorm);
  const double tiny = fmax(DBL_EPSILON * tnorm, DBL_MIN);
  __syncthreads();
  if (t == 0) {
    double di = s.d[0], ui = s.du[0];  // row i, as updated
    for (int i = 0; i < k - 1; ++i) {
      const double li = s.dl[i], dn = s.d[i + 1], un = s.du[i + 1];
      if (fabs(di) >= fabs(li)) {
        if (fabs(di) < tiny) di = di >= 0.0 ? tiny : -tiny;
        const double f = li / di;
        s.d[i] = di;
        s.du[i] = ui;
        s.dl[i] = f;
        s.piv[i] = 0;
        di = dn - f * ui;
        ui = un;
      } else {
        const double f = di / li;
        s.d[i] = li;
        s.du[i] = dn;
        s.du2[i] = un;
        s.dl[i] = f;
        s.piv[i] = 1;
        di = ui - f * dn;
        ui = -f * un;
      }
    }
    s.d[k - 1] = fabs(di) < tiny ? (di >= 0.0 ? tiny : -tiny) : di;
  }
  __syncthreads();
  for (int i = t; i < k; i += 64) s.d[i] = 1.0 / s.d[i];
  __syncthreads();
  for (int iter = 0; iter < 3; ++iter) {
    if (t == 0) {
      double xi = s.x[0];
#pragma unroll 4
      for (int i = 0; i < k - 1; ++i) {
        const double xn = s.x[i + 1], f = s.dl[i];
        const bool p = s.piv[i] != 0;
        const double top = p ? xn : xi, low = p ? xi : xn;
        s.x[i] = top;
        xi = low - f * top;
      }
      double x1 = xi * s.d[k - 1], x2 = 0.0;
      s.x[k - 1] = x1;
#pragma unroll 4
      for (int i = k - 2; i >= 0; --i) {
        const double v = ((s.x[i] - s.du2[i] * x2) - s.du[i] * x1) * s.d[i];
        s.x[i] = v;
        x2 = x1;
        x1 = v;
      }
    }
    __syncthreads();
    // by the largest entry, then to unit length: no square leaves the range
    double mx = 0.0, q = 0.0;
    for (int i = t; i < k; i += 64) mx = fmax(mx, fabs(s.x[i]));
    mx = wave_max(mx);
    for (int i = t; i < k; i += 64) {
      const double v = s.x[i] / mx;
      q += v * v;
    }
    const double inv = 1.0 / sqrt(wave_sum_all(q));
    for (int i = t; i < k; i += 64) s.x[i] = s.x[i] / mx * inv;
    __syncthreads();
  }
  // deterministic sign: largest-magnitude component (the first of equals) positive
  double mx = 0.0;
  for (int i = t; i < k; i += 64) mx = fmax(mx, fabs(s.x[i]));
  mx = wave_max(mx);
  unsigned long long at = 0;
  double sg = 1.0;
  for (int i0 = 0; i0 < k && at == 0; i0 += 64) {
    const double v = i0 + t < k ? s.x[i0 + t] : 0.0;
    at = __ballot(i0 + t < k && fabs(v) == mx);
    if (at) sg = __shfl(v, __ffsll((long long)at) - 1, 64) < 0.0 ? -1.0 : 1.0;
  }
  for (int i = t; i < k; i += 64) y[i] = sg * s.x[i];
}

// mode 0: convergence check (status[0] = stop, status[1] = niter; status may be
// host memory); mode 1: scal[3] = lowest eigenvalue, y = its vector.
__global__ __launch_bounds__(64) void k_tri(const double* alpha, const double* beta, int k, int mode,
                                           double beta_tol, double eig_tol, double eig_rel,
                                           double* scal, int* status, double* y) {
  __shared__ double ts[144], b2[144];
  __shared__ double as[128], bs[128];  // the tridiagonal, read once from HBM
  __shared__ TriWork work;
  const int t = threadIdx.x;
  for (int i = t; i < k; i += 64) {
    as[i] = alpha[i];
    bs[i] = mode == 0 || i < k - 1 ? beta[i] : 0.0;
  }
  __syncthreads();
  if (mode == 0) {  // check
    int bidx = -1;
    for (int j0 = 0; j0 < k && bidx < 0; j0 += 64) {
      const unsigned long long m = __ballot(j0 + t < k && bs[min(j0 + t, k - 1)] < beta_tol);
      if (m) bidx = j0 + __ffsll((long long)m) - 1;
    }
    if (bidx >= 0) {
      if (t == 0) { status[0] = 1; status[1] = bidx + 1; }
      return;
    }
    const double lam = k == 1 ? as[0] : tri_lowest(as, bs, k, ts, b2);
    if (t == 0) {
      scal[4] = lam;
      const double prev = scal[2];
      const bool stop = fabs(lam - prev) < fmax(eig_tol, eig_rel * fabs(lam));
      status[0] = stop;
      if (stop) status[1] = k;
      else scal[2] = lam;
    }
  } else {  // final
    const double lam = (k == 1) ? as[0] : tri_lowest(as, bs, k, ts, b2);
    if (t == 0) scal[3] = lam;
    if (k == 1) {
      if (t == 0) y[0] = 1.0;
    } else {
      tri_vector(as, bs, k, lam, y, work);
    }
  }
}

}  // namespace

namespace {
constexpr size_t LZ_ONE = 2 * NL;
// Every wave of a consuming kernel reads all partials of a sum, n / 4096 of them
// past 2^19 elements: work that grows with n^2.  Past LZ_PARTS a launch reduces
// them first (12 iterations, n = 2^21, 2^22, 2^23, 2^24, and 4 at 2^26: 2.79, 5.48,
// 14.6, 36.8 and 112 ms without, 2.78, 5.21, 13.6, 32.2 and 82 with 512; 256 and
// 1024 within 1 % of that but for 5.40 at 2^22 with 1024).
constexpr int LZ_PARTS = 512;
// Elements a thread holds: 1 to 2^18, 2 to 2^19, then 4.
int lz_elems(size_t n) { return n <= (size_t)256 * NL ? 1 : n <= (size_t)512 * NL ? 2 : 4; }
bool lz_one(size_t n) { return n <= LZ_ONE; }
}  // namespace

int lz_blocks(size_t n) { return std::max(1, (int)cdiv(n, (size_t)NL * lz_elems(n))); }

size_t lz_part_doubles(int kmax, size_t n) {
  // for every length up to n
  const size_t nb = std::max<size_t>(lz_blocks(n), std::min<size_t>(256, cdiv(std::max<size_t>(n, 1), NL)));
  return (2 * (size_t)kmax + 2) * nb;
}

void LzDev::alloc(int kmax_, size_t part_bytes_, size_t elem_bytes) {
  release();
  kmax = kmax_;
  part_bytes = part_bytes_;
  DMRG_HIP(hipMalloc(&alpha, kmax * sizeof(double)));
  DMRG_HIP(hipMalloc(&beta, kmax * sizeof(double)));
  DMRG_HIP(hipMalloc(&y, kmax * sizeof(double)));
  DMRG_HIP(hipMalloc(&scal, 8 * sizeof(double)));
  DMRG_HIP(hipMalloc(&part, part_bytes));
  DMRG_HIP(hipMalloc(&cvec, kmax * elem_bytes));
  DMRG_HIP(hipMemset(alpha, 0, kmax * sizeof(double)));
  DMRG_HIP(hipMemset(beta, 0, kmax * sizeof(double)));
}

void LzDev::release() {
  for (void* p : {(void*)alpha, (void*)beta, (void*)y, (void*)scal, part, cvec})
    if (p) (void)hipFree(p);
  alpha = beta = y = scal = nullptr;
  part = cvec = nullptr;
}

namespace {
// Partial-sum regions of LzDev::part (doubles): [0, nb) alpha, [nb, 2nb) norms,
// [2nb, ...) projection coefficients, (j*NC + c)*nb + blk.
inline double* partA(LzDev& d) { return (double*)d.part; }
inline double* partN(LzDev& d, int nb) { return (double*)d.part + nb; }
inline double* partC(LzDev& d, int nb) { return (double*)d.part + 2 * (size_t)nb; }
inline void need_parts(const LzDev& d, size_t n, int cnt) {
  const size_t need = (size_t)(cnt + 2) * lz_blocks(n) * sizeof(double);
  DMRG_REQUIRE(need <= d.part_bytes, "lanczos: partial buffer too small");
}

void totals(hipStream_t st, const double* part, int nb, int count, double* out) {
  if (nb <= LZ_PARTS)
    hipLaunchKernelGGL(k_totals<64>, dim3(count), dim3(64), 0, st, part, nb, out);
  else
    hipLaunchKernelGGL(k_totals<NL>, dim3(count), dim3(NL), 0, st, part, nb, out);
  DMRG_LAUNCH_CHECK();
}
// The sum of nb partials as every wave of the next kernel reads it: the partials
// themselves up to LZ_PARTS, past that one value (kept in `slot`).
Parts sum_of(hipStream_t st, const double* part, int nb, double* slot) {
  if (nb <= LZ_PARTS) return {part, nb};
  totals(st, part, nb, 1, slot);
  return {slot, 1};
}
}  // namespace

// Launch KERNEL<T, E> with the E of length n.
#define DMRG_LZ(KERNEL, ...)                                                                   \
  do {                                                                                         \
    const dim3 g_(lz_blocks(n)), b_(NL);                                                       \
    switch (lz_elems(n)) {                                                                     \
      case 1: hipLaunchKernelGGL((KERNEL<T, 1>), g_, b_, 0, st, __VA_ARGS__); break;           \
      case 2: hipLaunchKernelGGL((KERNEL<T, 2>), g_, b_, 0, st, __VA_ARGS__); break;           \
      default: hipLaunchKernelGGL((KERNEL<T, 4>), g_, b_, 0, st, __VA_ARGS__);                 \
    }                                                                                          \
    DMRG_LAUNCH_CHECK();                                                                       \
  } while (0)
// The same with one workgroup, n <= LZ_ONE.
#define DMRG_LZ_ONE(KERNEL, ...)                                                               \
  do {                                                                                         \
    const dim3 g_(1), b_(NL);                                                                  \
    if (n <= NL) hipLaunchKernelGGL((KERNEL<T, 1>), g_, b_, 0, st, __VA_ARGS__);               \
    else hipLaunchKernelGGL((KERNEL<T, 2>), g_, b_, 0, st, __VA_ARGS__);                       \
    DMRG_LAUNCH_CHECK();                                                                       \
  } while (0)

template <class T>
void lz_start(hipStream_t st, LzDev& d, T* theta, T* v0, size_t n, uint64_t seed, double thr) {
  if (lz_one(n)) {
    DMRG_LZ_ONE(k_one_start, theta, v0, n, seed, thr, d.scal);
    return;
  }
  const int nb = lz_blocks(n);
  need_parts(d, n, 0);
  DMRG_LZ(k_norm, theta, n, partN(d, nb), d.scal);
  const Parts first = sum_of(st, partN(d, nb), nb, d.scal + 5);
  DMRG_LZ(k_fill_small, theta, n, seed, thr, (const double*)partN(d, nb), first, partA(d));
  const Parts nrm = sum_of(st, partA(d), nb, d.scal + 5);
  DMRG_LZ(k_scale, v0, (const T*)theta, n, nrm, d.scal, (double*)nullptr, (double*)nullptr);
}

template <class T>
void fill_random(hipStream_t st, T* x, size_t n, uint64_t seed, uint64_t offset, double scale) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill_random<T>, dim3(std::min<size_t>(cdiv(n, NT), 2048)), dim3(NT), 0, st,
                     x, n, seed, offset, scale);
  DMRG_LAUNCH_CHECK();
}

template <class T>
void lz_step(hipStream_t st, LzDev& d, T* w, T* V, size_t n, int it, bool next) {
  DMRG_REQUIRE(it < d.kmax && it < 128, "lanczos: Krylov dimension exceeds 128");
  const int cnt = (it + 1) * Acc<T>::N;
  T* const vnext = next ? V + (size_t)(it + 1) * n : nullptr;
  if (lz_one(n)) {
    DMRG_LZ_ONE(k_one_step, (const T*)w, V, n, it, d.alpha, d.beta, d.scal, vnext);
    return;
  }
  need_parts(d, n, cnt);
  const int nb = lz_blocks(n);
  DMRG_LZ(k_alpha, (const T*)V + (size_t)it * n, (const T*)w, n, partA(d));
  const Parts al = sum_of(st, partA(d), nb, d.scal + 5);
  DMRG_LZ(k_sub_dots, w, (const T*)V, n, it, al, d.alpha, (const double*)d.beta, partC(d, nb));
  // every workgroup re-reduces the coefficients up to 256 partials each (n =
  // 2^18, 20 iterations: 6.3 us a time against 5.6 and 4.2 for a kernel of
  // its own); past that a wave per coefficient reduces them first
  const double* cv = nullptr;
  if (nb > 256) {
    totals(st, partC(d, nb), nb, cnt, (double*)d.cvec);
    cv = (const double*)d.cvec;
  }
  DMRG_LZ(k_orth_norm, w, (const T*)V, n, it, (const double*)partC(d, nb), cv, partN(d, nb));
  const Parts nrm = sum_of(st, partN(d, nb), nb, d.scal + 5);
  DMRG_LZ(k_scale, vnext, (const T*)w, n, nrm, d.scal, d.beta + it, (double*)nullptr);
}

template <class T>
void lz_dot(hipStream_t st, LzDev& d, const T* v, const T* w, size_t n) {
  need_parts(d, n, 0);
  DMRG_LZ(k_alpha, v, w, n, partA(d));
  totals(st, partA(d), lz_blocks(n), 1, d.alpha);
}

void lz_check(hipStream_t st, LzDev& d, int ncheck, double beta_tol, double eig_tol,
              double eig_rel, int* status) {
  DMRG_REQUIRE(ncheck <= 128, "lanczos: tridiagonal larger than 128");
  hipLaunchKernelGGL(k_tri, dim3(1), dim3(64), 0, st, d.alpha, d.beta, ncheck, 0, beta_tol, eig_tol,
                     eig_rel, d.scal, status, d.y);
  DMRG_LAUNCH_CHECK();
}

void lz_final(hipStream_t st, LzDev& d, int niter) {
  DMRG_REQUIRE(niter >= 1 && niter <= 128, "lanczos: bad Krylov dimension");
  hipLaunchKernelGGL(k_tri, dim3(1), dim3(64), 0, st, d.alpha, d.beta, niter, 1, 0.0, 0.0, 0.0,
                     d.scal, (int*)nullptr, d.y);
  DMRG_LAUNCH_CHECK();
}

template <class T>
void lz_ritz(hipStream_t st, LzDev& d, T* out, const T* V, size_t n, int niter, double* host) {
  DMRG_REQUIRE(niter <= 128, "lanczos: Krylov dimension exceeds 128");
  if (lz_one(n)) {
    DMRG_LZ_ONE(k_one_ritz, out, V, n, niter, (const double*)d.y, d.scal, host);
    return;
  }
  const int nb = lz_blocks(n);
  DMRG_LZ(k_ritz, out, V, n, niter, (const double*)d.y, partN(d, nb));
  const Parts nrm = sum_of(st, partN(d, nb), nb, d.scal + 5);
  DMRG_LZ(k_scale, out, (const T*)out, n, nrm, d.scal, (double*)nullptr, host);
}
#undef DMRG_LZ
#undef DMRG_LZ_ONE

#define DMRG_INST(T)                                                                             \
  template void lz_start<T>(hipStream_t, LzDev&, T*, T*, size_t, uint64_t, double);              \
  template void lz_step<T>(hipStream_t, LzDev&, T*, T*, size_t, int, bool);                      \
  template void lz_dot<T>(hipStream_t, LzDev&, const T*, const T*, size_t);                      \
  template void lz_ritz<T>(hipStream_t, LzDev&, T*, const T*, size_t, int, double*);             \
  template void fill_random<T>(hipStream_t, T*, size_t, uint64_t, uint64_t, double);
DMRG_INST(double)
DMRG_INST(cdouble)
#undef DMRG_INST

}  // namespace dmrg
