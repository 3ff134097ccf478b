// MFMA GEMM kernels for gfx950 (see gemm.hpp).
//
// Tile (the struct TileLoop) is the k-loop of every plain product and of the
// fused first H_eff step; k_gemm below it serves two-level operands only.
//
// What bounds these products on the card: FP64 MFMA at 64 cycles per
// 16x16x4 step (78.6 TF/s at 2.4 GHz, but a large FP64 product settles near
// 2.1 GHz, and lower the more operand traffic it causes), and everything a
// wave issues between two MFMAs.  Hence:
//  * operands travel in 16-byte chunks (2 FP64, 4 FP32, 1 complex128 value)
//    from memory to LDS to registers;
//  * the k-loop has no branch and no conditional load, so that the compiler
//    can count outstanding loads exactly: every load of a tile is issued with
//    its address clamped into the operand, and only the tiles that touch the
//    end of k (or, for an operand that is contiguous along its other index,
//    the end of that index) mask or shift what they got on the way to LDS;
//  * the memory instructions of one tile are interleaved with the MFMAs of
//    another: fragments of the next half tile are read while the present half
//    multiplies, also across the barrier (one per tile).
// Measured against the loop it replaces (element-wise LDS rows, loads under a
// branch, which made every wait a wait for all loads), us a call back to back:
// FP64 1024^3 48.4 -> 40.4 (A and B plain), 46.5 -> 37.9 (A transposed), 49.3 ->
// 41.1 (B transposed), 512^3 10.1 -> 9.0, 2048 x 512 x 2560 114 -> 94, 2560 x 2048 x
// 512 with A transposed 95 -> 85; FP32 the last two 83 -> 54 and 66 -> 51; complex
// 512^3 32.0 -> 21.2.
#include "gemm.hpp"

#include <type_traits>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <unordered_map>

namespace dmrg {
namespace {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

template <class T> struct GT;
// G1: accumulator register r of lane l holds output row (l/16) + 4r of the
// 16x16 block (f64 MFMA, group size 1); otherwise row 4(l/16) + r (f32 MFMA,
// group size 4).  Column = l % 16 in both cases.
template <> struct GT<double> { using E = double; using V4 = d4_t; static constexpr int P = 1; static constexpr bool G1 = true; };
template <> struct GT<cdouble> { using E = double; using V4 = d4_t; static constexpr int P = 2; static constexpr bool G1 = true; };
template <> struct GT<float> { using E = float; using V4 = f4_t; static constexpr int P = 1; static constexpr bool G1 = false; };

__device__ inline d4_t mfma(double a, double b, d4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline f4_t mfma(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <class T> __device__ inline void split(T v, typename GT<T>::E* out);
template <> __device__ inline void split<double>(double v, double* o) { o[0] = v; }
template <> __device__ inline void split<float>(float v, float* o) { o[0] = v; }
template <> __device__ inline void split<cdouble>(cdouble v, double* o) { o[0] = v.x; o[1] = v.y; }

template <class T> __device__ inline T conj_v(T v) { return conj(v); }
template <> __device__ inline float conj_v<float>(float v) { return v; }

// Two-level operand.
struct AddrTensor {
  View2 v;
  __device__ static long long dim(const Dim2& d, int i) {
    return (long long)(i % d.n1) * d.s1 + (long long)(i / d.n1) * d.s2;
  }
  __device__ long long operator()(int r, int c) const { return dim(v.row, r) + dim(v.col, c); }
};

typedef unsigned u4_t __attribute__((ext_vector_type(4)));

// The order of one half tile's instructions: after MFMA i of MH, its share of
// NR LDS reads (spread over the first half of the MFMAs) and of NX
// instructions of class MX (over the first half, or the second when X2).
template <int I, int MH, int NR, int MX, int NX, bool X2>
__device__ inline void interleave() {
  if constexpr (I < MH) {
    constexpr int h = MH / 2;
    constexpr int r = I < h ? NR * (I + 1) / h - NR * I / h : 0;
    constexpr int x = X2 ? (I >= h ? NX * (I - h + 1) / (MH - h) - NX * (I - h) / (MH - h) : 0)
                         : (I < h ? NX * (I + 1) / h - NX * I / h : 0);
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
    if constexpr (x > 0) __builtin_amdgcn_sched_group_barrier(MX, x, 0);
    interleave<I + 1, MH, NR, MX, NX, X2>();
  }
}
constexpr int kSchedDsWrite = 0x200, kSchedVmemRead = 0x20;

// One workgroup tile of C = op(A) op(B) over k in [kb, ke): WM x WN waves of
// FM x FN MFMA blocks of 16x16.  KFA / KFB: the operand is contiguous along k
// (A(m, k) at A[k + m lda], B(k, n) at B[k + n ldb]), otherwise along m / n.
// CA / CB conjugate.  VEC: 16-byte loads, which need the contiguous dimension
// to hold at least one chunk (any alignment); otherwise element loads.
//
// A k-tile is 128 bytes deep: eight chunks of VE values.  In LDS a k-contiguous
// operand is one 128-byte row per m (n), chunk c of row r at position
// c ^ (r % 8), so that the sixteen rows of a fragment read hit all banks; the
// other kind is one row of m (n) per k, padded by a chunk.  Lane (li, lk) =
// (lane % 16, lane / 16) holds, for MFMA e of half j, the value at
// k = (lk + 4j) VE + e: which four k an MFMA sums does not depend on the tile
// or on the operand's storage, so results depend on neither.  Real products
// add the two halves of every k-tile in accumulators of their own (CH = 2):
// two chains of half the length lose less to rounding (the split's
// first-order steps, which stop at 1e-14 |rho|, took 385 steps over 16 sweeps
// at chi = 256 against 737 with one chain).  An operand that
// is contiguous along m is read RV values of m at a time: MFMA block i of the
// wave then holds rows (i / RV) 16 RV + RV li + i % RV (row_of).
template <class T, bool CA, bool CB, bool KFA, bool KFB, int FM, int FN, int WM, int WN, bool VEC,
          int CH = GT<T>::P == 1 ? 2 : 1>
struct TileLoop {
  using V4 = typename GT<T>::V4;
  static constexpr int P = GT<T>::P, VE = 16 / sizeof(T), BK = 8 * VE;
  static constexpr int BM = 16 * FM * WM, BN = 16 * FN * WN, NT = 64 * WM * WN;
  static constexpr int RVA = FM % VE == 0 ? VE : (FM % 2 == 0 && VE >= 2 ? 2 : 1);
  static constexpr int RVB = FN % VE == 0 ? VE : (FN % 2 == 0 && VE >= 2 ? 2 : 1);
  static constexpr int NCA = BM * 8, NCB = BN * 8;  // chunks of one tile in memory
  static constexpr int NA = (NCA + NT - 1) / NT, NB = (NCB + NT - 1) / NT;
  // LDS chunks of one tile; every thread stores all its chunks, those past the
  // tile behind it
  static constexpr int SA = KFA ? NA * NT : BK * (BM / VE + 1);
  static constexpr int SB = KFB ? NB * NT : BK * (BN / VE + 1);
  static_assert((KFA || NCA % NT == 0) && (KFB || NCB % NT == 0), "chunks per thread");
  static constexpr int SMEM = 2 * (SA + SB);  // chunks of LDS
  using Acc = V4[P][FM][FN];
  struct Chunk { T v[VE]; };

  // row (column) of the wave's sub-tile that MFMA block i holds at lane index l
  __device__ static int row_of(bool kf, int rv, int i, int l) {
    return kf ? i * 16 + l : (i / rv) * 16 * rv + rv * l + i % rv;
  }

  // chunk c of an operand tile at (r0, k0); every address is in bounds
  template <bool KF, int ROWS>
  __device__ static u4_t load_chunk(const T* __restrict__ X, long long ld, int r0, int nr, int K,
                                    int k0, int c) {
    constexpr int NCH = KF ? 8 : ROWS / VE;
    const int lo = c % NCH, hi = c / NCH;
    const int x = (KF ? k0 : r0) + lo * VE, nx = KF ? K : nr;  // along the contiguous dimension
    const int y = min((KF ? r0 : k0) + hi, (KF ? nr : K) - 1);
    const T* p = X + (long long)y * ld;
    Chunk v;
    if constexpr (VEC) {
      __builtin_memcpy(&v, p + min(x, nx - VE), 16);
    } else {
#pragma unroll
      for (int q = 0; q < VE; ++q) v.v[q] = p[min(x + q, nx - 1)];
    }
    u4_t u;
    __builtin_memcpy(&u, &v, 16);
    return u;
  }
  // the chunk with values past the end of k zeroed, and those of a chunk that
  // was moved back into its row moved to their places
  template <bool KF, int ROWS>
  __device__ static u4_t mask_chunk(u4_t u, int r0, int nr, int K, int k0, int c) {
    constexpr int NCH = KF ? 8 : ROWS / VE;
    const int lo = c % NCH, hi = c / NCH;
    const int x = (KF ? k0 : r0) + lo * VE, nx = KF ? K : nr;
    const int back = VEC ? x - min(x, nx - VE) : 0;
    const bool in_k = KF || k0 + hi < K;
    Chunk v, w;
    __builtin_memcpy(&v, &u, 16);
#pragma unroll
    for (int q = 0; q < VE; ++q) {
      T y = v.v[q];
#pragma unroll
      for (int z = 1; z + q < VE; ++z) y = back == z ? v.v[q + z] : y;
      w.v[q] = (KF ? x + q < K : in_k) ? y : T(0);
    }
    __builtin_memcpy(&u, &w, 16);
    return u;
  }
  template <bool KF, int ROWS>
  __device__ static int slot_of(int c) {
    if constexpr (KF) return (c & ~7) | ((c ^ (c >> 3)) & 7);
    else return (c / (ROWS / VE)) * (ROWS / VE + 1) + c % (ROWS / VE);
  }
  template <bool CJ>
  __device__ static u4_t conj_chunk(u4_t u) {
    if constexpr (CJ && P == 2) u[3] ^= 0x80000000u;
    return u;
  }
  // fragments of half j of the tile in S, rows w0 .. w0 + 16 F
  template <bool KF, int F, int RV, int ROWS>
  __device__ static void read_frag(const u4_t* S, int w0, int j, int li, int lk, T (&f)[F][VE]) {
    if constexpr (KF) {
      const u4_t* p = S + (w0 + li) * 8 + ((lk + 4 * j) ^ (li & 7));
#pragma unroll
      for (int i = 0; i < F; ++i) {
        const u4_t u = p[16 * 8 * i];
        __builtin_memcpy(&f[i][0], &u, 16);
      }
    } else {
      const T* Sp = reinterpret_cast<const T*>(S) + w0 + RV * li;
#pragma unroll
      for (int e = 0; e < VE; ++e)
#pragma unroll
        for (int i = 0; i < F; i += RV) {
          T v[RV];
          __builtin_memcpy(v, __builtin_assume_aligned(
                                  Sp + ((lk + 4 * j) * VE + e) * (ROWS + VE) + 16 * i,
                                  RV * sizeof(T)), RV * sizeof(T));
#pragma unroll
          for (int q = 0; q < RV; ++q) f[i + q][e] = v[q];
        }
    }
  }

  // M, N, K: extents of the operands (K of the whole product: the last slice
  // ends there); the slice starts at a multiple of BK.  Returns with every
  // wave past its last LDS read (a barrier).
  __device__ static void run(u4_t* smem, int M, int N, int K, int kb, int ke, int m0, int n0,
                             const T* __restrict__ A, long long lda, const T* __restrict__ B,
                             long long ldb, Acc& acc) {
    u4_t(*As)[SA] = reinterpret_cast<u4_t(*)[SA]>(smem);
    u4_t(*Bs)[SB] = reinterpret_cast<u4_t(*)[SB]>(smem + 2 * SA);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave % WM, wn = wave / WM;
    const int li = lane & 15, lk = lane >> 4;
    u4_t ra[2][NA], rb[2][NB];  // two tiles in flight
    auto load = [&](int s, int k0) {
#pragma unroll
      for (int r = 0; r < NA; ++r)
        ra[s][r] = load_chunk<KFA, BM>(A, lda, m0, M, K, k0, NCA % NT ? min(t + r * NT, NCA - 1) : t + r * NT);
#pragma unroll
      for (int r = 0; r < NB; ++r)
        rb[s][r] = load_chunk<KFB, BN>(B, ldb, n0, N, K, k0, NCB % NT ? min(t + r * NT, NCB - 1) : t + r * NT);
    };
    auto store = [&](auto masked, int s, int k0, int buf) {
#pragma unroll
      for (int r = 0; r < NA; ++r) {
        const int c = t + r * NT;
        u4_t u = ra[s][r];
        if constexpr (decltype(masked)::value) u = mask_chunk<KFA, BM>(u, m0, M, K, k0, c);
        As[buf][slot_of<KFA, BM>(c)] = conj_chunk<CA>(u);
      }
#pragma unroll
      for (int r = 0; r < NB; ++r) {
        const int c = t + r * NT;
        u4_t u = rb[s][r];
        if constexpr (decltype(masked)::value) u = mask_chunk<KFB, BN>(u, n0, N, K, k0, c);
        Bs[buf][slot_of<KFB, BN>(c)] = conj_chunk<CB>(u);
      }
    };
    T fa[2][FM][VE], fb[2][FN][VE];
    auto read = [&](int slot, int buf, int j) {
      read_frag<KFA, FM, RVA, BM>(As[buf], wm * 16 * FM, j, li, lk, fa[slot]);
      read_frag<KFB, FN, RVB, BN>(Bs[buf], wn * 16 * FN, j, li, lk, fb[slot]);
    };
    V4 sum[CH][P][FM][FN];
    auto mul = [&](int slot) {
      auto& acc = sum[CH == 2 ? slot : 0];
#pragma unroll
      for (int e = 0; e < VE; ++e)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int n = 0; n < FN; ++n) {
            const T a = fa[slot][i][e], b = fb[slot][n][e];
            if constexpr (P == 1) {
              acc[0][i][n] = mfma(b, a, acc[0][i][n]);
            } else {
              acc[0][i][n] = mfma(b.x, a.x, acc[0][i][n]);
              acc[1][i][n] = mfma(b.y, a.x, acc[1][i][n]);
              acc[0][i][n] = mfma(-b.y, a.y, acc[0][i][n]);
              acc[1][i][n] = mfma(b.x, a.y, acc[1][i][n]);
            }
          }
    };
    // instructions of one half tile; FP32 is left to the compiler's own order
    // (measured: 55 us against 60 for 2560x2048x512)
    constexpr bool ORD = !std::is_same<T, float>::value;
    constexpr int MH = VE * FM * FN * (P == 2 ? 4 : 1);
    constexpr int NR = (KFA ? FM : VE * FM / RVA) + (KFB ? FN : VE * FN / RVB);
    constexpr int NL = (VEC ? 1 : VE) * (NA + NB);
    const int nk = (ke - kb + BK - 1) / BK;
    const int kl = kb + (nk - 1) * BK;  // last tile: later ones load it again, unused
    // Tile kt: its fragments are read half by half; tile kt + 1 goes to the
    // other LDS buffer, and the registers it leaves are loaded with kt + 3.
    auto body = [&](auto masked, auto uc, int kt) {
      constexpr int u = decltype(uc)::value;
      const int k0 = kb + kt * BK;
      read(1, u, 1);
      store(masked, u ^ 1, min(k0 + BK, kl), u ^ 1);
      mul(0);
      if constexpr (ORD) {
        interleave<0, MH, NR, kSchedDsWrite, NA + NB, false>();
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      read(0, u ^ 1, 0);
      mul(1);
      load(u ^ 1, min(k0 + 3 * BK, kl));
      if constexpr (ORD) {
        interleave<0, MH, NR, kSchedVmemRead, NL, true>();
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int n = 0; n < FN; ++n) sum[c][p][i][n] = V4{0, 0, 0, 0};
    std::integral_constant<int, 0> u0;
    std::integral_constant<int, 1> u1;
    load(0, kb);
    load(1, min(kb + BK, kl));
    store(std::true_type{}, 0, kb, 0);
    load(0, min(kb + 2 * BK, kl));
    __syncthreads();
    read(0, 0, 0);
    // tiles whose successor is neither the last one nor at an edge
    const bool edge = (!KFA && m0 + BM > M) || (!KFB && n0 + BN > N);
    const int free = edge ? 0 : nk - 2;
    int kt = 0;
    for (; kt + 2 <= free; kt += 2) {
      body(std::false_type{}, u0, kt);
      body(std::false_type{}, u1, kt + 1);
    }
    for (; kt + 2 <= nk; kt += 2) {
      body(std::true_type{}, u0, kt);
      body(std::true_type{}, u1, kt + 1);
    }
    if (kt < nk) body(std::true_type{}, u0, kt);
    __syncthreads();  // the last body read ahead
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int n = 0; n < FN; ++n) {
          acc[p][i][n] = sum[0][p][i][n];
          if constexpr (CH == 2) acc[p][i][n] += sum[CH - 1][p][i][n];
        }
  }
};

// 8 or 16 bytes at any multiple of 4.
template <int BYTES> struct RawOf;
template <> struct RawOf<16> { typedef unsigned type __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct RawOf<8> { typedef unsigned type __attribute__((ext_vector_type(2), aligned(4))); };

// C = alpha op(A) op(B) + beta C (plain operands).  Block z of the grid takes
// the k-slice [z Kc, z Kc + Kc) into C + z sC.  herm: a Hermitian product
// (M == N, BM == BN, beta == 0): only tiles on and above the diagonal are
// computed, each writes its conjugate mirror too.
template <class T, bool CA, bool CB, bool KFA, bool KFB, int FM, int FN, bool VEC>
__global__ __launch_bounds__(256) void k_tile(int M, int N, int K, int Kc, T alpha,
                                              const T* __restrict__ A, long long lda,
                                              const T* __restrict__ B, long long ldb, T beta,
                                              T* __restrict__ C, long long ldc, long long sC,
                                              int herm) {
  using TL = TileLoop<T, CA, CB, KFA, KFB, FM, FN, 2, 2, VEC>;
  __shared__ u4_t smem[TL::SMEM];
  if (herm && blockIdx.x > blockIdx.y) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int m0 = blockIdx.x * TL::BM, n0 = blockIdx.y * TL::BN;
  const int kb = blockIdx.z * Kc, ke = min(K, kb + Kc);
  typename TL::Acc acc;
  TL::run(smem, M, N, K, kb, ke, m0, n0, A, lda, B, ldb, acc);
  C += blockIdx.z * sC;
  const int li = lane & 15, lk = lane >> 4;
  const bool use_beta = !(real(beta) == 0.0 && imag(beta) == 0.0);
  // lane -> RW consecutive rows of C (the MFMA blocks of one group, see row_of),
  // register r -> column lk + 4r (f64) or 4 lk + r (f32)
  constexpr int RW = KFA ? 1 : TL::RVA;
#pragma unroll
  for (int i = 0; i < FM; i += RW)
#pragma unroll
    for (int n = 0; n < FN; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + wm * 16 * FM + TL::row_of(KFA, TL::RVA, i, li);
        const int gn = n0 + wn * 16 * FN +
                       TL::row_of(KFB, TL::RVB, n, GT<T>::G1 ? lk + 4 * r : 4 * lk + r);
        if (gm < M && gn < N) {
          T v[RW];
#pragma unroll
          for (int q = 0; q < RW; ++q) {
            if constexpr (TL::P == 1) v[q] = T(acc[0][i + q][n][r]);
            else v[q] = make_scalar<T>(acc[0][i + q][n][r], acc[1][i + q][n][r]);
            v[q] = alpha * v[q];
          }
          const long long idx = gm + (long long)gn * ldc;
          if constexpr (RW == 1) {
            if (use_beta) v[0] = v[0] + beta * C[idx];
            C[idx] = v[0];
          } else if (gm + RW <= M) {  // one access for the RW rows
            using R = typename RawOf<RW * sizeof(T)>::type;
            R u;
            if (use_beta) {
              T old[RW];
              u = *reinterpret_cast<const R*>(C + idx);
              __builtin_memcpy(old, &u, sizeof(old));
#pragma unroll
              for (int q = 0; q < RW; ++q) v[q] = v[q] + beta * old[q];
            }
            __builtin_memcpy(&u, v, sizeof(v));
            *reinterpret_cast<R*>(C + idx) = u;
          } else {
#pragma unroll
            for (int q = 0; q < RW; ++q)
              if (gm + q < M) {
                if (use_beta) v[q] = v[q] + beta * C[idx + q];
                C[idx + q] = v[q];
              }
          }
          if (herm && blockIdx.x != blockIdx.y)
#pragma unroll
            for (int q = 0; q < RW; ++q)
              if (gm + q < M) C[gn + (long long)(gm + q) * ldc] = conj_v(v[q]);
        }
      }
}

// ---------------------------------------------------------------------------
// Two-level operands (gemm_tensor).
// Workgroup: 256 threads = 4 wave64s in a 2x2 grid, each owning a
// (BM/2) x (BN/2) sub-tile of 16x16 MFMA blocks; operand tiles of depth BK are
// staged through LDS (double buffered, one-element row padding), with the
// global loads of the next PF tiles issued before the MFMAs of the current one.
// ---------------------------------------------------------------------------
template <class T, int BM, int BN, int BK>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, T alpha,
                                              const T* __restrict__ A, AddrTensor aa,
                                              const T* __restrict__ B, AddrTensor ab, T beta,
                                              T* __restrict__ C, AddrTensor ac) {
  using E = typename GT<T>::E;
  using V4 = typename GT<T>::V4;
  constexpr int P = GT<T>::P;
  constexpr int NT = 256, PF = 2;
  constexpr int PADM = BM + 1, PADN = BN + 1;
  constexpr int FM = BM / 32, FN = BN / 32;  // 16x16 blocks per wave
  constexpr int NA = BM * BK / NT, NB = BN * BK / NT;

  __shared__ E As[2][P][BK][PADM];
  __shared__ E Bs[2][P][BK][PADN];

  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;

  T ra[PF][NA], rb[PF][NB];

  auto idxA = [&](int r, int& m, int& k) {
    m = t % BM;
    k = t / BM + r * (NT / BM);
  };
  auto idxB = [&](int r, int& n, int& k) {
    k = t % BK;
    n = t / BK + r * (NT / BK);
  };
  // register stage `s` <- operand tiles at depth k0; a tile inside all three
  // bounds loads without per-element checks (one branch for the whole stage)
  const bool inner_mn = m0 + BM <= M && n0 + BN <= N;
  auto load = [&](int s, int k0) {
    if (inner_mn && k0 + BK <= K) {
#pragma unroll
      for (int r = 0; r < NA; ++r) {
        int m, k;
        idxA(r, m, k);
        ra[s][r] = A[aa(m0 + m, k0 + k)];
      }
#pragma unroll
      for (int r = 0; r < NB; ++r) {
        int n, k;
        idxB(r, n, k);
        rb[s][r] = B[ab(k0 + k, n0 + n)];
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      int m, k;
      idxA(r, m, k);
      int gm = m0 + m, gk = k0 + k;
      ra[s][r] = (gm < M && gk < K) ? A[aa(gm, gk)] : T(0);
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      int n, k;
      idxB(r, n, k);
      int gn = n0 + n, gk = k0 + k;
      rb[s][r] = (gn < N && gk < K) ? B[ab(gk, gn)] : T(0);
    }
  };
  // LDS buffer `buf` <- register stage `s`
  auto store = [&](int s, int buf) {
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      int m, k;
      idxA(r, m, k);
      E e[P];
      split<T>(ra[s][r], e);
#pragma unroll
      for (int p = 0; p < P; ++p) As[buf][p][k][m] = e[p];
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      int n, k;
      idxB(r, n, k);
      E e[P];
      split<T>(rb[s][r], e);
#pragma unroll
      for (int p = 0; p < P; ++p) Bs[buf][p][k][n] = e[p];
    }
  };

  V4 acc[P][FM][FN];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[p][i][j] = V4{0, 0, 0, 0};

  const int nk = (K + BK - 1) / BK;
  const int li = lane & 15, lk = lane >> 4;
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      E af[P][FM], bf[P][FN];
#pragma unroll
      for (int p = 0; p < P; ++p) {
#pragma unroll
        for (int i = 0; i < FM; ++i) af[p][i] = As[buf][p][kk + lk][wm * (BM / 2) + i * 16 + li];
#pragma unroll
        for (int j = 0; j < FN; ++j) bf[p][j] = Bs[buf][p][kk + lk][wn * (BN / 2) + j * 16 + li];
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          if constexpr (P == 1) {
            acc[0][i][j] = mfma(bf[0][j], af[0][i], acc[0][i][j]);
          } else {
            acc[0][i][j] = mfma(bf[0][j], af[0][i], acc[0][i][j]);
            acc[0][i][j] = mfma(-bf[1][j], af[1][i], acc[0][i][j]);
            acc[1][i][j] = mfma(bf[1][j], af[0][i], acc[1][i][j]);
            acc[1][i][j] = mfma(bf[0][j], af[1][i], acc[1][i][j]);
          }
        }
    }
  };
  // PF register stages: tile j travels in stage j % PF, then LDS buffer
  // j & 1.  While tile kt is multiplied, tiles kt+1 .. kt+PF are in flight
  // (kt+PF issued into the stage that tile kt just left); tile kt+1 is then
  // staged into the other LDS buffer.  The loop is unrolled by PF so that
  // stage indices are compile-time constants.
  load(0, 0);
  store(0, 0);
#pragma unroll
  for (int s = 1; s < PF; ++s)
    if (s < nk) load(s, s * BK);
  __syncthreads();
  for (int kt = 0; kt < nk; kt += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int tile = kt + u;
      if (tile >= nk) break;
      const int buf = (PF % 2 == 0) ? (u & 1) : (tile & 1);  // kt is even when PF is
      if (tile + PF < nk) load(u, (tile + PF) * BK);
      compute(buf);
      if (tile + 1 < nk) store((u + 1) % PF, buf ^ 1);
      __syncthreads();
    }
  }

  // Epilogue: lane -> row li of C; register r -> column lk + 4r (f64) or
  // 4*lk + r (f32) of each 16x16 block.
  const bool use_beta = !(real(beta) == 0.0 && imag(beta) == 0.0);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int gm = m0 + wm * (BM / 2) + i * 16 + li;
        int gn = n0 + wn * (BN / 2) + j * 16 + (GT<T>::G1 ? lk + 4 * r : 4 * lk + r);
        if (gm < M && gn < N) {
          T v;
          if constexpr (P == 1) v = T(acc[0][i][j][r]);
          else v = make_scalar<T>(acc[0][i][j][r], acc[1][i][j][r]);
          v = alpha * v;
          long long idx = ac(gm, gn);
          if (use_beta) v = v + beta * C[idx];
          C[idx] = v;
        }
      }
}


// One launch: `slices` slices of Kc (a multiple of the k-tile depth when there
// is more than one).
template <class T, bool CA, bool CB, bool KFA, bool KFB>
void launch(hipStream_t st, GemmTile tl, int M, int N, int K, int Kc, int slices, T alpha,
            const T* A, int lda, const T* B, int ldb, T beta, T* C, int ldc, long long sC,
            int herm) {
#define DMRG_TILE(FM_, FN_, VEC_)                                                              \
  hipLaunchKernelGGL((k_tile<T, CA, CB, KFA, KFB, FM_, FN_, VEC_>),                            \
                     dim3(cdiv(M, 32 * FM_), cdiv(N, 32 * FN_), slices), dim3(256), 0, st, M, N, \
                     K, Kc, alpha, A, (long long)lda, B, (long long)ldb, beta, C,              \
                     (long long)ldc, sC, herm)
  // 16-byte loads need one whole chunk along each operand's contiguous
  // dimension (2 FP64, 4 FP32, 1 complex128 value); the products that do not
  // have it, at the ends of a chain, are tiny
  constexpr int VE = 16 / (int)sizeof(T);
  if constexpr (VE > 1) {
    if ((KFA ? K : M) < VE || (KFB ? K : N) < VE) {
      DMRG_TILE(1, 1, false);
      DMRG_LAUNCH_CHECK();
      return;
    }
  }
  if (tl.bm == 32) DMRG_TILE(1, 1, true);
  else if (tl.bn == 32) DMRG_TILE(2, 1, true);
  else DMRG_TILE(2, 2, true);
#undef DMRG_TILE
  DMRG_LAUNCH_CHECK();
}

template <class T>
void dispatch(hipStream_t st, int opA, int opB, GemmTile tl, int M, int N, int K, int Kc,
              int slices, T alpha, const T* A, int lda, const T* B, int ldb, T beta, T* C, int ldc,
              long long sC, int herm) {
  const bool ta = op_trans(opA), tb = op_trans(opB);
  bool ca = op_conj(opA), cb = op_conj(opB);
  if (!is_cplx<T>::value) ca = cb = false;
  constexpr int MAX_COLS = 65535 * 32;  // grid.y of the narrowest tile
  if (N > MAX_COLS && !herm) {
    for (int n0 = 0; n0 < N; n0 += MAX_COLS)
      dispatch<T>(st, opA, opB, tl, M, std::min(MAX_COLS, N - n0), K, Kc, slices, alpha, A, lda,
                  B + (tb ? (long long)n0 : (long long)n0 * ldb), ldb, beta,
                  C + (long long)n0 * ldc, ldc, sC, 0);
    return;
  }
#define DMRG_P4(TA_, TB_, CA_, CB_) \
  launch<T, CA_, CB_, TA_, !TB_>(st, tl, M, N, K, Kc, slices, alpha, A, lda, B, ldb, beta, C, ldc, sC, herm)
  if (!ca && !cb) {
    if (!ta && !tb) DMRG_P4(false, false, false, false);
    else if (!ta && tb) DMRG_P4(false, true, false, false);
    else if (ta && !tb) DMRG_P4(true, false, false, false);
    else DMRG_P4(true, true, false, false);
  } else {
    if constexpr (is_cplx<T>::value) {
      int code = (ta ? 8 : 0) | (tb ? 4 : 0) | (ca ? 2 : 0) | (cb ? 1 : 0);
      switch (code) {
        case 1: DMRG_P4(false, false, false, true); break;
        case 2: DMRG_P4(false, false, true, false); break;
        case 3: DMRG_P4(false, false, true, true); break;
        case 5: DMRG_P4(false, true, false, true); break;
        case 6: DMRG_P4(false, true, true, false); break;
        case 7: DMRG_P4(false, true, true, true); break;
        case 9: DMRG_P4(true, false, false, true); break;
        case 10: DMRG_P4(true, false, true, false); break;
        case 11: DMRG_P4(true, false, true, true); break;
        case 13: DMRG_P4(true, true, false, true); break;
        case 14: DMRG_P4(true, true, true, false); break;
        default: DMRG_P4(true, true, true, true); break;
      }
    }
  }
#undef DMRG_P4
}

// ---------------------------------------------------------------------------
// Tile autotuner.  When enabled (gemm_autotune), the first call of each (scalar
// type, ops, M, N, K, Hermitian) shape times the 32x32, 64x32 (not for a
// Hermitian product) and 64x64 tiles on the caller's stream, drained first (one
// warm-up each, then four interleaved rounds of one launch each into a scratch
// output, keeping each tile's fastest), and keeps the fastest for the rest of the
// process -- the caller's tile unless another is at least 3 % faster; later calls
// of that shape use it.  All tiles sum over k in the same order, so tuning never
// changes a result: runs are bit-reproducible across processes.  A call made
// while its stream is being captured into a graph uses the caller's tile and
// records nothing.
// ---------------------------------------------------------------------------
struct TuneKey {
  int dt, opA, opB, M, N, K, herm;
  bool operator==(const TuneKey& o) const {
    return dt == o.dt && opA == o.opA && opB == o.opB && M == o.M && N == o.N && K == o.K &&
           herm == o.herm;
  }
};
struct TuneKeyHash {
  size_t operator()(const TuneKey& k) const {
    uint64_t h = 1469598103934665603ull;
    for (int v : {k.dt, k.opA, k.opB, k.M, k.N, k.K, k.herm}) {
      h ^= (uint64_t)(uint32_t)v;
      h *= 1099511628211ull;
    }
    return (size_t)h;
  }
};
std::mutex g_tune_mu;
std::unordered_map<TuneKey, GemmTile, TuneKeyHash> g_tune;
std::atomic<int> g_tune_on{0};
// DMRG_GEMM_AUTOTUNE_LOG=1 prints each tuning decision (shape, candidate
// times, choice) to stderr.
const bool g_tune_log = [] {
  const char* v = std::getenv("DMRG_GEMM_AUTOTUNE_LOG");
  return v && v[0] == '1';
}();
constexpr int kTuneDevices = 64;
void* g_tune_buf[kTuneDevices] = {};
size_t g_tune_cap[kTuneDevices] = {};

template <class T> constexpr int dt_code() { return is_cplx<T>::value ? 1 : (std::is_same<T, float>::value ? 2 : 0); }

template <class T>
GemmTile tuned_tile(hipStream_t st, int opA, int opB, GemmTile tl, int M, int N, int K,
                    const T* A, int lda, const T* B, int ldb, int herm) {
  const TuneKey key{dt_code<T>(), opA, opB, M, N, K, herm};
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_tune.find(key);
  if (it != g_tune.end()) return it->second;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  DMRG_HIP(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone) return tl;
  int dev = 0;
  DMRG_HIP(hipGetDevice(&dev));
  DMRG_REQUIRE(dev >= 0 && dev < kTuneDevices, "gemm autotune: device ordinal out of range");
  const size_t bytes = (size_t)M * N * sizeof(T);
  if (g_tune_cap[dev] < bytes) {
    if (g_tune_buf[dev]) DMRG_HIP(hipFree(g_tune_buf[dev]));
    g_tune_buf[dev] = nullptr;
    g_tune_cap[dev] = 0;
    DMRG_HIP(hipMalloc(&g_tune_buf[dev], bytes));
    g_tune_cap[dev] = bytes;
  }
  T* Cs = static_cast<T*>(g_tune_buf[dev]);
  hipEvent_t e0, e1;
  DMRG_HIP(hipEventCreate(&e0));
  DMRG_HIP(hipEventCreate(&e1));
  constexpr int ROUNDS = 4;
  const GemmTile cand[3] = {{32, 32}, {64, 64}, {64, 32}};
  const int NC = herm ? 2 : 3;
  float t_min[3] = {0.f, 0.f, 0.f};
  GemmTile best = tl;
  float best_ms = 1e30f;
  try {
    // Not the device: draining that is refused while any thread captures a
    // stream of it, and breaks the capture.
    DMRG_HIP(hipStreamSynchronize(st));
    for (int c = 0; c < NC; ++c)  // warm-up: code and operands into the caches
      dispatch<T>(st, opA, opB, cand[c], M, N, K, K, 1, T(1), A, lda, B, ldb, T(0), Cs, M, 0, herm);
    // Rounds interleave the candidates, and each keeps its fastest launch,
    // so work that other streams run meanwhile biases no candidate.
    for (int r = 0; r < ROUNDS; ++r)
      for (int c = 0; c < NC; ++c) {
        DMRG_HIP(hipEventRecord(e0, st));
        dispatch<T>(st, opA, opB, cand[c], M, N, K, K, 1, T(1), A, lda, B, ldb, T(0), Cs, M, 0,
                    herm);
        DMRG_HIP(hipEventRecord(e1, st));
        DMRG_HIP(hipEventSynchronize(e1));
        float ms = 0.f;
        DMRG_HIP(hipEventElapsedTime(&ms, e0, e1));
        t_min[c] = r == 0 ? ms : std::min(t_min[c], ms);
      }
    // the caller's tile stands unless another is at least 3 % faster
    for (int c = 0; c < NC; ++c)
      if (cand[c].bm == tl.bm && cand[c].bn == tl.bn) best_ms = t_min[c];
    for (int c = 0; c < NC; ++c)
      if (t_min[c] < 0.97f * best_ms) {
        best_ms = t_min[c];
        best = cand[c];
      }
    if (g_tune_log)
      std::fprintf(stderr,
                   "[gemm autotune] dt %d op %d%d%s M %d N %d K %d: 32x32 %.1f, 64x64 %.1f, "
                   "64x32 %.1f us -> %dx%d\n",
                   key.dt, opA, opB, herm ? " herm" : "", M, N, K, 1e3f * t_min[0],
                   1e3f * t_min[1], 1e3f * t_min[2], best.bm, best.bn);
  } catch (...) {
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    throw;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  g_tune.emplace(key, best);
  return best;
}

template <class T>
void plain(hipStream_t st, int opA, int opB, GemmTile tl, int M, int N, int K, T alpha, const T* A,
           int lda, const T* B, int ldb, T beta, T* C, int ldc, int herm) {
  DMRG_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gemm: negative size");
  DMRG_REQUIRE(opA >= 0 && opA <= 3 && opB >= 0 && opB <= 3, "gemm: bad op");
  if (M == 0 || N == 0) return;
  DMRG_REQUIRE(K >= 1, "gemm: empty sum");
  if (g_tune_on.load(std::memory_order_relaxed))
    tl = tuned_tile<T>(st, opA, opB, tl, M, N, K, A, lda, B, ldb, herm);
  dispatch<T>(st, opA, opB, tl, M, N, K, K, 1, alpha, A, lda, B, ldb, beta, C, ldc, 0, herm);
}

}  // namespace

void gemm_autotune(bool on) { g_tune_on.store(on ? 1 : 0); }
int gemm_autotune_entries() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  return (int)g_tune.size();
}

namespace {
// Cycles (at 2.1 GHz) of one k-tile on a CU that holds w workgroups of the
// grid, from FP64 products with K = 1024 and 8192 (MFMA alone: 1024, 512 and
// 256 cycles per workgroup).  A single workgroup is bound by its own chain of
// barrier and LDS reads, several by the MFMAs and, for the small tiles, by the
// lower clock that their operand traffic leaves.  Complex k-tiles hold the same
// bytes and twice the MFMAs; their 64x64 tile pays from two workgroups a CU on
// (2048 x 2048 x 1024: 486 us, 514 with 32x32; 1024 x 1024 x 1024 137 and 135, x 32
// 13.0 and 12.0), the 64x32 one too (640 x 640 x 1024: 79 us, 72 with 32x32; 1152 x
// 1152 x 1024 194 and 196; first step of the matvec at 256, d = 5: 602 us in all, 606).
double tile_cycles(const GemmTile& t, int w, bool cplx) {
  if (cplx) {
    if (t.bm == 32) return 640.0 * w;
    return t.bn == 32 ? std::max(1320.0, 1200.0 * w) : std::max(2620.0, 2360.0 * w);
  }
  if (t.bm == 32) return std::max(430.0, 332.0 * w);
  if (t.bn == 32) return std::max(620.0, 610.0 * w);
  return std::max(1250.0, 1050.0 * w);
}
constexpr int kCUs = 256;
inline int per_cu(const GemmTile& t, int M, int N, int slices) {
  const long long tiles = (long long)cdiv(M, t.bm) * cdiv(N, t.bn) * slices;
  return (int)((tiles + kCUs - 1) / kCUs);
}
GemmTile pick_square(int N, bool cplx) {
  const GemmTile a{32, 32}, b{64, 64};
  return tile_cycles(a, per_cu(a, N, N, 1), cplx) < tile_cycles(b, per_cu(b, N, N, 1), cplx) ? a : b;
}
}  // namespace

// The tile with the fewest modelled cycles; they agree with the measured order
// on the sweep's shapes (us for 64x64, 64x32, 32x32: 1024^3 44, 43, 46;
// 512^3 21, 12.5, 9.3; 1280x1024x256 24, 19, 17; 2560x2048x512 98, 105, 109).
GemmTile gemm_pick_tile(int M, int N, int K, bool complex_) {
  (void)K;
  GemmTile best{64, 64};
  double c = tile_cycles(best, per_cu(best, M, N, 1), complex_);
  for (const GemmTile t : {GemmTile{64, 32}, GemmTile{32, 32}}) {
    const double ct = tile_cycles(t, per_cu(t, M, N, 1), complex_);
    if (ct < c) {
      c = ct;
      best = t;
    }
  }
  return best;
}

namespace {
// One thread per row r: C(r, :) = A(r, :) B with B (K x N, column-major),
// K <= KM and N <= 32.  B sits in LDS zero-padded to KM rows, so the unrolled
// k-loop needs no bounds; the operand column offsets are tabulated once per
// workgroup and each thread does one div/mod pair per operand row.
template <class T, int KM>
__global__ __launch_bounds__(256) void k_rows_small(int M, int N, int K, const T* __restrict__ A,
                                                    View2 va, const T* __restrict__ B,
                                                    T* __restrict__ C, View2 vc) {
  __shared__ T Bs[KM * 32];
  __shared__ long long ca[KM], cc[32];
  for (int e = threadIdx.x; e < KM * 32; e += 256) {
    const int k = e % KM, j = e / KM;
    Bs[e] = (k < K && j < N) ? B[k + (size_t)K * j] : T(0);
  }
  for (int k = threadIdx.x; k < KM; k += 256) ca[k] = k < K ? AddrTensor::dim(va.col, k) : 0;
  for (int j = threadIdx.x; j < N; j += 256) cc[j] = AddrTensor::dim(vc.col, j);
  __syncthreads();
  for (int r = blockIdx.x * 256 + threadIdx.x; r < M; r += gridDim.x * 256) {
    const long long ra = AddrTensor::dim(va.row, r), rc = AddrTensor::dim(vc.row, r);
    T x[KM];
#pragma unroll
    for (int k = 0; k < KM; ++k) x[k] = k < K ? A[ra + ca[k]] : T(0);
    for (int j = 0; j < N; ++j) {
      T y = T(0);
#pragma unroll
      for (int k = 0; k < KM; ++k) y = y + x[k] * Bs[k + KM * j];
      C[rc + cc[j]] = y;
    }
  }
}
}  // namespace

namespace {
// ---------------------------------------------------------------------------
// Split-BF16 FP32 GEMM: C = A B with every FP32 operand written as
// hi + mid + lo, three bf16 numbers (round to nearest even, then the exact FP32
// residual, rounded again), so together they carry 24 significand bits.  The
// six products hi*hi, hi*mid, mid*hi, hi*lo, lo*hi, mid*mid (the ones above
// 2^-24 relative) run on v_mfma_f32_16x16x32_bf16 with FP32 accumulation; the
// result has FP32-class accuracy.  hi*hi goes to its own accumulator.
//
// MFMA operand layout (gfx950, checked with random integer inputs): lane l
// holds row l%16 of the left operand and column l%16 of the right one, over
// the eight consecutive k = 8*(l/16) .. +7; result register r is row
// 4*(l/16)+r, column l%16.  B is passed in the left slot, so the result is
// C^T per lane: lane l -> row l%16 of C, register r -> column 4*(l/16)+r.
//
// A(m, k) = A[k + m*lda] (KFA) or A[m + k*lda]; B(k, n) = B[k + n*ldb] (KFB)
// or B[n + k*ldb]; C column-major.  64x64 workgroup tile, 2x2 waves of 32x32,
// BK = 32, LDS rows of 40 bf16 (80 B: 16-byte aligned, no bank conflicts for
// the 16 rows of one 128-bit read).
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
constexpr int BF_BK = 32, BF_LD = 40;

// x = hi + mid + lo: the float -> bf16 casts compile to gfx950's
// v_cvt_pk_bf16_f32 (round to nearest even, two values per instruction), the
// bf16 -> float ones to a shift.
__device__ inline void split3(float x, unsigned short& h, unsigned short& m, unsigned short& l) {
  const __bf16 bh = (__bf16)x;
  const float r1 = x - (float)bh;
  const __bf16 bm = (__bf16)r1;
  const __bf16 bl = (__bf16)(r1 - (float)bm);
  memcpy(&h, &bh, 2);
  memcpy(&m, &bm, 2);
  memcpy(&l, &bl, 2);
}

// blockIdx.z is the slice of Kc values of k (a multiple of BK); its product goes
// to C + z zstride.  The loads have no branch and run two k-tiles ahead: row
// indices past the operand are clamped (those results are not stored), a chunk
// past the last whole k-tile is the last one again, and the remainder of K is a
// tile of its own behind the loop.  A branch around a load makes every wait of
// the loop a wait for all of them: 1556 x 451 x 2255 with odd leading
// dimensions took 124 us with checked scalar loads one tile ahead on 200
// workgroups, 52 + 6 us in four slices now (1945 x 1804 x 389: 72 -> 40).
struct __attribute__((packed, aligned(4))) F4u {
  float v[4];
};
template <bool KFA, bool KFB>
__global__ __launch_bounds__(256) void k_gemm_bf3(int M, int N, int K, int Kc,
                                                  const float* __restrict__ A, long long lda,
                                                  const float* __restrict__ B, long long ldb,
                                                  float* __restrict__ C, long long ldc,
                                                  long long zstride) {
  constexpr int BM = 64, BN = 64;  // 8 elements of A and of B per thread
  __shared__ __attribute__((aligned(16))) unsigned short As[2][3][BM][BF_LD];
  __shared__ __attribute__((aligned(16))) unsigned short Bs[2][3][BN][BF_LD];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  const int kb = blockIdx.z * Kc, ke = min(K, kb + Kc);
  C += blockIdx.z * zstride;
  // Thread t holds 8 consecutive k of one row (one 16-byte LDS store per bf16
  // plane): k-fast operand row t/4, k = 8 (t%4) (two 16-byte loads); m-fast
  // operand row t%64, k = 8 (t/64) (eight loads, each of 64 rows).
  const int rowA = KFA ? t >> 2 : lane, kqA = KFA ? (t & 3) * 8 : wave * 8;
  const int rowB = KFB ? t >> 2 : lane, kqB = KFB ? (t & 3) * 8 : wave * 8;
  const int ga = min(m0 + rowA, M - 1), gb = min(n0 + rowB, N - 1);
  const float* const pA = KFA ? A + ga * lda + kqA : A + ga + kqA * lda;
  const float* const pB = KFB ? B + gb * ldb + kqB : B + gb + kqB * ldb;
  auto load_op = [](bool kfast, const float* __restrict__ X, long long ld, int k0, float (&r)[8]) {
    if (kfast) {
      const F4u u = *reinterpret_cast<const F4u*>(X + k0);
      const F4u v = *reinterpret_cast<const F4u*>(X + k0 + 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] = u.v[q], r[q + 4] = v.v[q];
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) r[q] = X[(long long)(k0 + q) * ld];
    }
  };
  // the remainder: k0 + q + kq < ke only
  auto load_tail = [&](bool kfast, const float* __restrict__ X, long long ld, int k0, int kq,
                       float (&r)[8]) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const bool in = k0 + kq + q < ke;
      const int k = in ? k0 + q : ke - 1 - kq;
      const float v = X[kfast ? (long long)k : (long long)k * ld];
      r[q] = in ? v : 0.f;
    }
  };
  auto store_op = [](unsigned short (*S)[BM][BF_LD], int row, int kq, const float (&r)[8]) {
    unsigned short h[8], mi[8], lo[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) split3(r[q], h[q], mi[q], lo[q]);
    uint4 v;
    memcpy(&v, h, 16);
    *reinterpret_cast<uint4*>(&S[0][row][kq]) = v;
    memcpy(&v, mi, 16);
    *reinterpret_cast<uint4*>(&S[1][row][kq]) = v;
    memcpy(&v, lo, 16);
    *reinterpret_cast<uint4*>(&S[2][row][kq]) = v;
  };
  f4_t acc_hh[2][2], acc_x[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc_hh[i][j] = acc_x[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
  const int li = lane & 15, lg = lane >> 4;
  auto compute = [&](int buf) {
    bf8_t af[2][3], bfr[2][3];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        af[i][p] = *reinterpret_cast<const bf8_t*>(&As[buf][p][wm * 32 + i * 16 + li][lg * 8]);
        bfr[i][p] = *reinterpret_cast<const bf8_t*>(&Bs[buf][p][wn * 32 + i * 16 + li][lg * 8]);
      }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        acc_hh[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j][0], af[i][0], acc_hh[i][j], 0, 0, 0);
        f4_t x = acc_x[i][j];
        x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j][1], af[i][1], x, 0, 0, 0);
        x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j][0], af[i][2], x, 0, 0, 0);
        x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j][2], af[i][0], x, 0, 0, 0);
        x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j][0], af[i][1], x, 0, 0, 0);
        x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j][1], af[i][0], x, 0, 0, 0);
        acc_x[i][j] = x;
      }
  };
  const int nf = (ke - kb) / BF_BK;  // whole k-tiles
  if (nf > 0) {
    float ra[2][8], rb[2][8];
    auto load = [&](int kt, int s) {
      const int k0 = kb + min(kt, nf - 1) * BF_BK;
      load_op(KFA, pA, lda, k0, ra[s]);
      load_op(KFB, pB, ldb, k0, rb[s]);
    };
    auto store = [&](int s) {
      store_op(As[s], rowA, kqA, ra[s]);
      store_op(Bs[s], rowB, kqB, rb[s]);
    };
    load(0, 0);
    load(1, 1);
    store(0);
    load(2, 0);
    __syncthreads();
    // two tiles a pass, so that registers and buffers have fixed indices
    for (int kt = 0; kt + 1 < nf; kt += 2) {
      compute(0);
      store(1);
      load(kt + 3, 1);
      __syncthreads();
      compute(1);
      store(0);
      load(kt + 4, 0);
      __syncthreads();
    }
    if (nf & 1) compute(0);
  }
  const int kt0 = kb + nf * BF_BK;
  if (kt0 < ke) {
    float xa[8], xb[8];
    load_tail(KFA, pA, lda, kt0, kqA, xa);
    load_tail(KFB, pB, ldb, kt0, kqB, xb);
    __syncthreads();  // the last whole tile has been read
    store_op(As[0], rowA, kqA, xa);
    store_op(Bs[0], rowB, kqB, xb);
    __syncthreads();
    compute(0);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + wm * 32 + i * 16 + li;
        const int gn = n0 + wn * 32 + j * 16 + lg * 4 + r;
        if (gm < M && gn < N) C[gm + (long long)gn * ldc] = acc_hh[i][j][r] + acc_x[i][j][r];
      }
}
}  // namespace

namespace {
// C[i] = sum_{z<S} W[i + z*stride] for i < M*N over an M x N block (ld ldc);
// fixed summation order (deterministic).
// FP32 partials into an FP64 result (TO = double, T = float): the sum is
// formed in FP32 as for an FP32 result, then widened and multiplied by
// s1 * s2 (each taken as 1 when not positive), the factor that undoes the
// unit-max scaling of the FP32 operands.
template <class T, class TO>
__global__ void k_splitk_sum(const T* __restrict__ W, int S, long long stride, int M, int N,
                             TO* __restrict__ C, int ldc, const double* __restrict__ s1,
                             const double* __restrict__ s2) {
  double f = 1.0;
  if constexpr (!std::is_same<T, TO>::value) {
    const double a = *s1, b = *s2;
    f = (a > 0.0 ? a : 1.0) * (b > 0.0 ? b : 1.0);
  }
  const long long tot = (long long)M * N;
  const bool packed = ldc == M;  // C contiguous: no row/column split per element
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < tot;
       e += (long long)gridDim.x * blockDim.x) {
    T v = W[e];
    for (int z = 1; z < S; ++z) v = v + W[e + z * stride];
    const long long o = packed ? e : (e % M) + (e / M) * (long long)ldc;
    if constexpr (std::is_same<T, TO>::value) C[o] = v;
    else C[o] = (TO)v * f;
  }
}

template <class T, class TO>
bool splitk_impl(hipStream_t st, int opA, int opB, int M, int N, int K, const T* A, int lda,
                 const T* B, int ldb, TO* C, int ldc, T* ws, size_t ws_elems, const double* s1,
                 const double* s2) {
  // Slices of whole k-tiles in one launch.  The number of slices and the tile
  // are those with the fewest modelled cycles: the k-tiles of one slice, the
  // start and end of a workgroup, and the pass that sums the partial products
  // (5.5 TB/s and 2 us for its launch; 2048 x 512 x 2560 in FP64: one slice 108
  // us, two 93 + 6, four 88 + 9).
  constexpr int BK = 128 / (int)sizeof(T);
  const int nkt = (int)cdiv(K, BK);
  const GemmTile tiles[3] = {{64, 64}, {64, 32}, {32, 32}};
  GemmTile tile{64, 64};
  int S = 1;
  double best = 1e300;
  bool was_long = false;
  for (int sl : {1, 2, 3, 4, 6, 8, 12, 16}) {
    if (sl > 1 && ((size_t)sl * M * N > ws_elems || nkt < 4 * sl)) break;
    // FP32: a slice sums at most 768 values per accumulator (two per slice)
    // where the workspace allows it, however many slices are fastest
    const bool long_sum = std::is_same<T, float>::value && K > 2 * 768 * sl;
    const double per = (double)cdiv(nkt, sl);
    const double sum =
        sl == 1 ? 0.0 : 2.1e9 * (2e-6 + ((double)sl * sizeof(T) + sizeof(TO)) * M * N / 5.5e12);
    for (const GemmTile& t : tiles) {
      const double c = (per + 3.0) * tile_cycles(t, per_cu(t, M, N, sl), is_cplx<T>::value) + sum;
      if (c < best || (was_long && !long_sum)) {
        best = c;
        S = sl;
        tile = t;
        was_long = long_sum;
      }
    }
  }
  if (S == 1) return false;
  const int Kc = (int)cdiv(nkt, S) * BK;
  S = (int)cdiv(K, Kc);  // no empty slice
  dispatch<T>(st, opA, opB, tile, M, N, K, Kc, S, T(1), A, lda, B, ldb, T(0), ws, M,
              (long long)M * N, 0);
  const long long tot = (long long)M * N;
  hipLaunchKernelGGL((k_splitk_sum<T, TO>),
                     dim3((unsigned)std::min<long long>(cdiv(tot, 256), 4096)), dim3(256), 0, st,
                     (const T*)ws, S, (long long)M * N, M, N, C, ldc, s1, s2);
  DMRG_LAUNCH_CHECK();
  return true;
}
}  // namespace

void gemm_f32_split_bf16(hipStream_t st, int opA, int opB, int M, int N, int K, const float* A,
                         int lda, const float* B, int ldb, float* C, int ldc, float* ws,
                         size_t ws_elems) {
  DMRG_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gemm_bf16x3: negative size");
  DMRG_REQUIRE(opA >= 0 && opA <= 3 && opB >= 0 && opB <= 3, "gemm_bf16x3: bad op");
  if (M == 0 || N == 0) return;
  // op(A) (m, k): transposed storage is k-fast; op(B) (k, n): plain storage is k-fast
  const bool kfa = op_trans(opA), kfb = !op_trans(opB);
  // Slices of k, each of eight k-tiles or more, up to three workgroups a CU: two
  // are resident (LDS), and a grid just past that ends in a nearly empty wave
  // (out-step at 768 x 768, D = 5, 576 tiles: matvec 386 us unsliced, 354 with two
  // slices; limits of 256 to 1024 workgroups are within 8 % of one another at
  // fourteen other shapes, in either direction).
  const int nkt = (int)cdiv(K, BF_BK);
  const long long tiles = (long long)cdiv(M, 64) * cdiv(N, 64);
  int S = 1;
  if (ws)
    while (S < 16 && tiles * S < 768 && nkt >= 8 * (S + 1) && (size_t)(S + 1) * M * N <= ws_elems)
      ++S;
  const int Kc = std::max(1, (int)cdiv(nkt, S)) * BF_BK;
  S = std::max(1, (int)cdiv(K, Kc));  // no empty slice
  const dim3 grid(cdiv(M, 64), cdiv(N, 64), S);
  float* const out = S > 1 ? ws : C;
  const long long ldo = S > 1 ? M : ldc, zs = S > 1 ? (long long)M * N : 0;
#define DMRG_BF3(KA_, KB_)                                                                        \
  hipLaunchKernelGGL((k_gemm_bf3<KA_, KB_>), grid, dim3(256), 0, st, M, N, K, Kc, A,              \
                     (long long)lda, B, (long long)ldb, out, ldo, zs)
  if (kfa && kfb) DMRG_BF3(true, true);
  else if (kfa) DMRG_BF3(true, false);
  else if (kfb) DMRG_BF3(false, true);
  else DMRG_BF3(false, false);
#undef DMRG_BF3
  if (S > 1)
    hipLaunchKernelGGL((k_splitk_sum<float, float>),
                       dim3((unsigned)std::min<long long>(cdiv((size_t)M * N, 256), 4096)),
                       dim3(256), 0, st, (const float*)ws, S, (long long)M * N, M, N, C, ldc,
                       (const double*)nullptr, (const double*)nullptr);
  DMRG_LAUNCH_CHECK();
}

template <class T>
bool gemm_splitk(hipStream_t st, int opA, int opB, int M, int N, int K, const T* A, int lda,
                 const T* B, int ldb, T* C, int ldc, T* ws, size_t ws_elems) {
  return splitk_impl<T, T>(st, opA, opB, M, N, K, A, lda, B, ldb, C, ldc, ws, ws_elems, nullptr,
                           nullptr);
}

bool gemm_nn_splitk_to_f64(hipStream_t st, int M, int N, int K, const float* A, int lda,
                           const float* B, int ldb, double* C, int ldc, float* ws,
                           size_t ws_elems, const double* s1, const double* s2) {
  return splitk_impl<float, double>(st, OP_N, OP_N, M, N, K, A, lda, B, ldb, C, ldc, ws, ws_elems,
                                    s1, s2);
}

namespace {
// First step of the two-site H_eff with the MPO-bond step applied in the
// epilogue (d = 2, real scalars).  The workgroup computes the tile of
// X = L^T theta with rows (w + D a') for 16 consecutive a' (all D values of w)
// and columns (ss + 4 b) for 16 consecutive b (all four ss): wave j owns the
// columns 16 j .. 16 j + 15, four b, and all D row blocks.  The finished tile
// changes lanes through LDS inside each wave, and lane (a', b) contracts its
// 4D values with WW into the 4D outputs Y[a' + cL ss' + 4 cL b + 4 cL cR n],
// summing over c = w + D ss in order.  WW is the same for every lane and comes
// through scalar loads.  X never reaches HBM.
// MFMA-bound; LDS is held to 40 KB for D <= 5, four workgroups a CU: the 1024
// tiles of cL = cR = 512 are then resident at once.
template <class T, int D, bool VEC>
__global__ __launch_bounds__(256) void k_heff2_x_mpo(int cL, int cR, const T* __restrict__ Lenv,
                                                     const T* __restrict__ theta,
                                                     const T* __restrict__ WW,
                                                     T* __restrict__ Y) {
  constexpr int DD = 4, K2 = D * DD, BM = 16 * D;
  // a second accumulator chain only where the registers leave room for it
  constexpr int CH = sizeof(T) == 4 || D <= 3 ? 2 : 1;
  using TL = TileLoop<T, false, false, true, true, D, 1, 1, 4, VEC, CH>;
  constexpr int XC = 16 * (int)sizeof(T) / 16;  // chunks of a row of one wave's 16 columns
  constexpr int XS = 4 * BM * XC;
  __shared__ u4_t smem[TL::SMEM > XS ? TL::SMEM : XS];
  const int lane = threadIdx.x & 63, wn = threadIdx.x >> 6;
  typename TL::Acc acc;
  // A(m, k) = Lenv[k + m cL], B(k, n) = theta[k + n cL]
  TL::run(smem, D * cL, DD * cR, cL, 0, cL, blockIdx.x * BM, blockIdx.y * 64, Lenv, cL, theta, cL,
          acc);
  const int li = lane & 15, lk = lane >> 4;
  // value (row, ss + 4 bq) of the wave's block at T index of chunk
  // (column / VE) ^ (row % XC): the sixteen rows of a store spread over banks
  T* const xw = reinterpret_cast<T*>(smem + wn * BM * XC);
  auto at = [&](int row, int col) {
    return row * 16 + (((col / TL::VE) ^ (row & (XC - 1))) * TL::VE) + col % TL::VE;
  };
#pragma unroll
  for (int i = 0; i < D; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      xw[at(i * 16 + li, GT<T>::G1 ? lk + 4 * r : 4 * lk + r)] = acc[0][i][0][r];
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  const int a = blockIdx.x * 16 + li, b = blockIdx.y * 16 + wn * 4 + lk;
  if (a >= cL || b >= cR) return;
  T x[K2];
#pragma unroll
  for (int w = 0; w < D; ++w)
#pragma unroll
    for (int ss = 0; ss < DD; ++ss) x[w + D * ss] = xw[at(w + D * li, ss + DD * lk)];
  T* const yb = Y + a + (size_t)cL * DD * b;
  const size_t sn = (size_t)cL * DD * cR;
  // the constant address space: nothing in the launch writes WW, and past a
  // barrier the compiler would load it into vector registers otherwise
  typedef const T __attribute__((address_space(4))) ConstT;
  const ConstT* const Wc = (const ConstT*)(uintptr_t)WW;
#pragma unroll 1
  for (int n = 0; n < D; ++n)
#pragma unroll
    for (int sp = 0; sp < DD; ++sp) {
      const ConstT* const wc = Wc + K2 * (sp + DD * n);
      T y = T(0);
#pragma unroll
      for (int c = 0; c < K2; ++c) y = y + x[c] * wc[c];
      yb[(size_t)cL * sp + sn * n] = y;
    }
}
}  // namespace

template <class T>
bool heff2_x_mpo(hipStream_t st, int cL, int cR, int d, int D, const T* Lenv, const T* theta,
                 const T* WW, T* Y) {
  if constexpr (is_cplx<T>::value) {
    return false;
  } else {
    if (d != 2 || D < 2 || D > 8 || cL < 1 || cR < 1) return false;
    const dim3 grid(cdiv(cL, 16), cdiv(cR, 16));
    const bool vec = cL >= 16 / (int)sizeof(T);  // both operands are contiguous along cL
    switch (D) {
#define DMRG_XM(D_)                                                                             \
  case D_:                                                                                      \
    if (vec)                                                                                    \
      hipLaunchKernelGGL((k_heff2_x_mpo<T, D_, true>), grid, dim3(256), 0, st, cL, cR, Lenv,    \
                         theta, WW, Y);                                                         \
    else                                                                                        \
      hipLaunchKernelGGL((k_heff2_x_mpo<T, D_, false>), grid, dim3(256), 0, st, cL, cR, Lenv,   \
                         theta, WW, Y);                                                         \
    break
      DMRG_XM(2); DMRG_XM(3); DMRG_XM(4); DMRG_XM(5); DMRG_XM(6); DMRG_XM(7); DMRG_XM(8);
#undef DMRG_XM
      default: return false;
    }
    DMRG_LAUNCH_CHECK();
    return true;
  }
}

template <class T>
bool gemm_rows_small(hipStream_t st, int M, int N, int K, const T* A, View2 va, const T* B, T* C,
                     View2 vc) {
  if (K > 32 || N > 32 || K < 1) return false;
  if (M == 0 || N == 0) return true;
  const unsigned grid = (unsigned)std::min<long long>(cdiv(M, 256), 8192);
  if (K <= 16)
    hipLaunchKernelGGL((k_rows_small<T, 16>), dim3(grid), dim3(256), 0, st, M, N, K, A, va, B, C, vc);
  else if (K <= 24)
    hipLaunchKernelGGL((k_rows_small<T, 24>), dim3(grid), dim3(256), 0, st, M, N, K, A, va, B, C, vc);
  else
    hipLaunchKernelGGL((k_rows_small<T, 32>), dim3(grid), dim3(256), 0, st, M, N, K, A, va, B, C, vc);
  DMRG_LAUNCH_CHECK();
  return true;
}

template <class T>
void gemm(hipStream_t st, int opA, int opB, int M, int N, int K, T alpha, const T* A, int lda,
          const T* B, int ldb, T beta, T* C, int ldc, GemmTile tile) {
  plain<T>(st, opA, opB, tile, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, 0);
}

template <class T>
void gemm_herm(hipStream_t st, int opA, int opB, int N, int K, T alpha, const T* A, int lda,
               const T* B, int ldb, T* C, int ldc, GemmTile tile) {
  if (tile.bm != tile.bn) tile = pick_square(N, is_cplx<T>::value);  // mirrored tile by tile
  plain<T>(st, opA, opB, tile, N, N, K, alpha, A, lda, B, ldb, T(0), C, ldc, 1);
}

template <class T>
void gemm_tensor(hipStream_t st, int M, int N, int K, T alpha, const T* A, View2 va, const T* B,
                 View2 vb, T beta, T* C, View2 vc, GemmTile tile) {
  DMRG_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gemm_tensor: negative size");
  if (M == 0 || N == 0) return;
  // 32x32 tiles serve grids that cannot fill the chip with 64x64 ones
  constexpr int BK = is_cplx<T>::value ? 16 : 32;
  const AddrTensor aa{va}, ab{vb}, ac{vc};
  if (tile.bm == 32)
    hipLaunchKernelGGL((k_gemm<T, 32, 32, BK>), dim3(cdiv(M, 32), cdiv(N, 32)), dim3(256), 0, st, M,
                       N, K, alpha, A, aa, B, ab, beta, C, ac);
  else
    hipLaunchKernelGGL((k_gemm<T, 64, 64, 16>), dim3(cdiv(M, 64), cdiv(N, 64)), dim3(256), 0, st, M,
                       N, K, alpha, A, aa, B, ab, beta, C, ac);
  DMRG_LAUNCH_CHECK();
}

#define DMRG_INST(T)                                                                         \
  template void gemm<T>(hipStream_t, int, int, int, int, int, T, const T*, int, const T*, int, \
                        T, T*, int, GemmTile);                                                 \
  template void gemm_herm<T>(hipStream_t, int, int, int, int, T, const T*, int, const T*, int,  \
                             T*, int, GemmTile);                                                \
  template void gemm_tensor<T>(hipStream_t, int, int, int, T, const T*, View2, const T*, View2, \
                               T, T*, View2, GemmTile);                                        \
  template bool gemm_rows_small<T>(hipStream_t, int, int, int, const T*, View2, const T*, T*,  \
                                   View2);                                                      \
  template bool gemm_splitk<T>(hipStream_t, int, int, int, int, int, const T*, int, const T*,   \
                               int, T*, int, T*, size_t);                                       \
  template bool heff2_x_mpo<T>(hipStream_t, int, int, int, int, const T*, const T*, const T*, T*);
DMRG_INST(double)
DMRG_INST(cdouble)
DMRG_INST(float)
#undef DMRG_INST


}  // namespace dmrg
