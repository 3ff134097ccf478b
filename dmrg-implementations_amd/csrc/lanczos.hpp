// Lanczos building blocks (replaces the rocBLAS dot/axpy/gemv/nrm2/scal
// sequence and the rocsolver_dsteqr calls of the reference's
// lanczos_eigensolver, gpu-rocm/dmrg2-gpu/src/dmrg2_gpu_impl.h:970-1160, and
// the scalar kernels of gpu-rocm/common/scalar_traits.h:422-489).
//
// Reductions carry no atomics or fences: every workgroup of a vector kernel
// writes one partial sum, and the next kernel in the stream reduces the
// partials (each of its workgroups, in the same fixed order), so results are
// deterministic and bit-identical across workgroups.
#pragma once
#include "common.hpp"

namespace dmrg {

struct LzDev {
  // device scalars / small arrays
  double* alpha = nullptr;     // [kmax]
  double* beta = nullptr;      // [kmax]
  double* y = nullptr;         // [kmax] Ritz coefficients
  double* scal = nullptr;      // [8]: 0 norm, 1 inv, 2 prev_energy, 3 energy, 4 check value, 5 sum of partials
  void* part = nullptr;        // partial sums (bytes), lz_part_doubles(kmax, n) doubles
  void* cvec = nullptr;        // [kmax] projection coefficients (T)
  int kmax = 0;
  size_t part_bytes = 0;
  void alloc(int kmax_, size_t part_bytes_, size_t elem_bytes);
  void release();
};

// Number of workgroups used by the vector kernels for length n.
int lz_blocks(size_t n);
// Size of LzDev::part, in doubles, for Krylov dimension kmax and length n.
size_t lz_part_doubles(int kmax, size_t n);

// Start of a Lanczos call: theta, overwritten with the splitmix64 stream `seed`
// (U[-1,1)) when |theta| < thr; v0 = theta / |theta| (0 when |theta| <= 1e-300);
// prev_energy := 1e30.
template <class T> void lz_start(hipStream_t st, LzDev& d, T* theta, T* v0, size_t n, uint64_t seed,
                                 double thr);
// What follows w = H v_it in iteration it (V: the basis, n apart):
// alpha[it] = <v_it, w>;  w -= alpha[it] v_it + beta[it-1] v_{it-1};
// w -= sum_{j <= it} <v_j, w> v_j;  beta[it] = |w|;  v_{it+1} = w / beta[it] if
// `next` (0 when beta[it] <= 1e-300).  w is scratch afterwards.
template <class T> void lz_step(hipStream_t st, LzDev& d, T* w, T* V, size_t n, int it, bool next);
// alpha[0] = Re <v, w>
template <class T> void lz_dot(hipStream_t st, LzDev& d, const T* v, const T* w, size_t n);
// Convergence check on T(ncheck) (every third iteration).
// Converged when |E - E_prev| < max(eig_tol, eig_rel |E|).  status[0] = stop,
// status[1] = niter when it stops; pinned host memory, read after the stream.
void lz_check(hipStream_t st, LzDev& d, int ncheck, double beta_tol, double eig_tol,
              double eig_rel, int* status);
// Lowest eigenpair of T(niter) -> scal[3], y.
void lz_final(hipStream_t st, LzDev& d, int niter);
// out = V y / |V y| (niter columns; 0 when |V y| <= 1e-300); host[0] = |V y|,
// host[3] = scal[3] (pinned host memory).
template <class T> void lz_ritz(hipStream_t st, LzDev& d, T* out, const T* V, size_t n, int niter,
                                double* host);

// Fill `x` with entries scale*U[-1,1) from the splitmix64 stream `seed`,
// starting at stream position `offset` (complex: two outputs per entry).
template <class T> void fill_random(hipStream_t st, T* x, size_t n, uint64_t seed, uint64_t offset,
                                    double scale);

}  // namespace dmrg
