// FP64, one matrix per workgroup: orders 33..96, the fused eigendecomposition of
// whole batches and lists, the stage entries, and the roots entry's Schur form;
// and the orders below where this beats the lane groups (few_matrices).
//
// One matrix per workgroup, two kernels:
//
//   k_reduce<CAP, W>   the Hessenberg reduction on a dense LDS tile
//                      (reduce_block); for the fused path its compact form
//                      goes to the V and E planes, which serve as workspace;
//                      for the stages also Q (hessenberg, zunghr).
//   k_schur<SL, NT>    one wavefront (chain_wave) runs the QR iteration on the
//                      banded tile (lahqr_stream), the others hold the Schur vectors in
//                      registers, NT lanes per row, and replay the recorded
//                      sweeps (SchurRows); then the eigenvector solve and
//                      V = Z X on the matrix cores.
//
// Segments: the row of a Schur vector is cut in two, of 16 to 32 columns up to
// order 64 (three or four wavefronts per SIMD), of 40 or 48 above (two, which
// the LDS of 60 to 90 KB per workgroup leaves in any case): half the wavefronts,
// and less ring, than four segments of 20 or 24 (3,328 matrices: order 65 24.4
// -> 22.4 ms, 79 34.4 -> 31.6, 88 45.7 -> 39.0).  Up to 24 columns the allocation
// is held to four wavefronts per SIMD although that spills (order 48 x 8,192:
// 12.3 -> 11.5 ms), at 32 columns to three.  LDS is allocated for the batch's
// order: 40 KB at n = 64 (four matrices per CU), 71 KB at n = 88 (two).
//
// Measured, whole passes (in brackets the kernels these replaced, whose bulge
// chase went through LDS): order 64 x 65,536 182 ms (371; reduction 25,
// k_schur 153 in a trace), order 79 x 3,328 31.6 ms (233: a workgroup barrier per
// half step and Z in global memory; reduction 3.6, k_schur 27.9), the
// stages hessenberg + zlahqr + ztrevc at order 40 x 2,048 3.1 ms (21).  What
// bounds order 64 is instruction issue, the chain wavefront's (7,700 steps of
// about 88 instructions and 230 sweeps of about 480 more per matrix) and,
// on the same SIMDs, the Schur vectors'.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "veig_stream.hpp"

using namespace veig;

namespace {

struct BigArgs {
  double *rA, *iA;  // A / H / T
  double *rB, *iB;  // V / Q / Z / R
  double *rE, *iE;  // E / tau
  int32_t *info;
  Geom G;
  int itmax;
  uint32_t flags;
  const int32_t *list, *list_count;  // fused: only these matrices
  const double *rC, *iC;             // roots: the coefficients
};

// the matrix of this workgroup, from the batch or the list (whose length is
// only known on the device: the workgroups past it find none)
__device__ __forceinline__ bool block_matrix(const BigArgs &a, int64_t &m) {
  if (a.list) {
    const int64_t cnt = *a.list_count, b = blockIdx.x;
    m = b < cnt ? a.list[xcd_remap(b, cnt)] : 0;
    return b < cnt;
  }
  m = xcd_block();
  return m < a.G.nmat;
}

// ---------------------------------------------------------------------------
// reduction
// ---------------------------------------------------------------------------
enum { RD_FUSED = 0, RD_GEHRD = 1, RD_HESS = 2, RD_UNGHR = 3, RD_BANDED = 4 };  // (banded: for k_qr_band)

// (at most three wavefronts per SIMD at capacity 24: four, which zunghr's registers
// allow, took 1.23 ms instead of 0.75 at 65,536 matrices of order 24 in tiles of 64,
// whose lines the workgroups in flight then push out of the L2, and 69 us instead
// of 57 at 4,096)
template <int CAP, int W, int MODE>
__global__ __launch_bounds__((ReduceBlock<CAP, W>::kThreads)) __attribute__((amdgpu_waves_per_eu(1, CAP == 24 ? 3 : 8)))
void k_reduce(BigArgs a) {
  using S = ReduceBlock<CAP, W>;
  extern __shared__ double2 lds[];
  S &sm = *reinterpret_cast<S *>(lds);
  double2 *tau = lds + sizeof(S) / sizeof(double2);
  int64_t m;
  if (!block_matrix(a, m)) return;  // workgroup-uniform
  const int n = a.G.n, tid = threadIdx.x, r = tid % CAP, q = tid / CAP;
  const int64_t base = a.G.mat_base(m), vb = a.G.vec_base(m);
  unsigned top = 0;
  if constexpr (MODE == RD_UNGHR) {
    top = reduce_load(sm, n, a.G, base, a.rA, a.iA, [&]() -> unsigned {
      if (tid + 1 >= n) return 0u;
      const cx<double> t = mk<double>(a.rE[vb + a.G.ve(tid)], a.iE[vb + a.G.ve(tid)]);
      st<double>(tau + tid, t);
      return high_word(t) >= kNonFinite ? kNonFinite : 0u;
    });
  } else {
    top = reduce_load(sm, n, a.G, base, a.rA, a.iA, [] { return 0u; });
    const int e = reduce_block<MODE != RD_BANDED>(sm, n, top, tau);
    const bool fused = MODE == RD_FUSED || MODE == RD_BANDED;
    reduce_store(sm, n, a.G, base, fused ? a.rB : a.rA, fused ? a.iB : a.iA, e);
    if (a.rE && tid + 1 < n) {
      const cx<double> t = ld<double>(tau + tid);
      a.rE[vb + a.G.ve(tid)] = t.re;
      a.iE[vb + a.G.ve(tid)] = t.im;
    }
  }
  if constexpr (MODE == RD_HESS || MODE == RD_UNGHR) {
    double *re = MODE == RD_HESS ? a.rB : a.rA, *im = MODE == RD_HESS ? a.iB : a.iA;
    if (__builtin_expect(top >= kNonFinite, 0)) {
      form_q_rare(sm, n, tau, a.G, base, re, im);
      return;
    }
    cx<double> z[S::CH];
    form_q_block(sm, n, tau, z);
#pragma unroll
    for (int j = 0; j < S::CH; ++j) {
      const int c = q * S::CH + j;
      if (q < W && r < n && c < n) {
        const int64_t idx = base + a.G.el(r, c);
        re[idx] = z[j].re;
        im[idx] = z[j].im;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// QR iteration, Schur vectors, eigenvectors
// ---------------------------------------------------------------------------
enum { SC_FUSED = 0, SC_LAHQR = 1, SC_TREVC = 2, SC_ROOTS = 3 };

template <int SL, int NT>
constexpr int schur_threads() {
  constexpr int RW = SchurRows<SL, NT>::RW;
  return 64 * (1 + (SL * NT + RW - 1) / RW);
}

// wavefronts per SIMD the register allocation is held to
template <int SL>
constexpr int schur_waves() { return SL <= 24 ? 4 : (SL <= 32 ? 3 : 2); }

template <int SL, int NT, int MODE>
__global__ __launch_bounds__((schur_threads<SL, NT>())) __attribute__((amdgpu_waves_per_eu(schur_waves<SL>()))) void k_schur(BigArgs a) {
  using Rows = SchurRows<SL, NT>;
  using Ring = typename Rows::Ring;
  constexpr int CAP = Rows::CAP, P = (CAP + 63) / 64;
  extern __shared__ double2 lds[];
  Ring &ring = *reinterpret_cast<Ring *>(lds);
  const BandTile t{MODE == SC_TREVC ? lds : lds + sizeof(Ring) / sizeof(double2)};
  int64_t m;
  if (!block_matrix(a, m)) return;  // workgroup-uniform
  const int n = a.G.n, lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), zw = (blockDim.x >> 6) - 1;
  const int64_t base = a.G.mat_base(m), vb = a.G.vec_base(m);
  // the band (Hessenberg part, or upper triangle) from memory, by every wavefront
  for (int i = threadIdx.x; i < BandTile::entries(n); i += blockDim.x) st<double>(t.h + i, mk<double>(0, 0));
  __syncthreads();
  if constexpr (MODE == SC_ROOTS) {
    // the companion matrix of c_0 + ... + c_n x^n (create_companion_matrices,
    // Toolbox.hpp:605-643): ones below the diagonal, -c_r / c_n in the last
    // column (Smith's division)
    const int64_t cb = a.G.vec_base(m, 1) + (m / a.G.T) * a.G.T;  // slots of n + 1 entries
    const cx<double> lead = mk<double>(a.rC[cb + n * a.G.T], a.iC[cb + n * a.G.T]);
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
      const cx<double> c = cdiv(mk<double>(a.rC[cb + r * a.G.T], a.iC[cb + r * a.G.T]), lead);
      if (r >= 1) st<double>(t.at(r, r - 1), mk<double>(1, 0));
      st<double>(t.at(r, n - 1), mk(-c.re, -c.im));
    }
  } else {
    const double *re = MODE == SC_FUSED ? a.rB : a.rA, *im = MODE == SC_FUSED ? a.iB : a.iA;
    constexpr int sub = MODE == SC_TREVC ? 0 : 1;
    for (int c = threadIdx.x >> 6; c < n; c += zw + 1)
      for (int r = lane; r <= c + sub && r < n; r += 64) {
        const int64_t idx = base + a.G.el(r, c);
        st<double>(t.at(r, c), mk<double>(re[idx], im[idx]));
      }
  }
  int hw = 0;  // the wavefront of the iteration; zi: this one among the others
  if constexpr (MODE == SC_TREVC) __syncthreads();
  else hw = chain_wave(ring.simd);
  const int zi = w < hw ? w : w - 1;
  if (w == hw) {
    // ---------------- the iteration and the eigenvector solve ----------------
    const unsigned top = wave_top(t.h, BandTile::entries(n), lane);
    if (MODE == SC_LAHQR && lane == 0) ring.rare = top >= kNonFinite;  // (read after the next barrier)
    const int e2 = scale_exponent(top);  // (eigenvectors do not depend on it)
    if (__builtin_expect(e2 != 0, 0)) scale_entries(t.h, BandTile::entries(n), lane, 64, e2);
    lds_order();
    __builtin_amdgcn_s_setprio(3);  // the workgroup waits for the chain: it issues first on its SIMD
    if constexpr (MODE != SC_TREVC) {
      if constexpr (MODE == SC_LAHQR) {
        make_subdiag_real(t, n, lane, &ring.step[1][0].c);
        __syncthreads();  // its phases are out
      }
      const int nfail = lahqr_stream<P, true>(t, n, lane, ring, a.itmax);
      for (int r = lane; r < n; r += 64) {
        const cx<double> e = cldexp(ld<double>(t.at(r, r)), e2);
        a.rE[vb + a.G.ve(r)] = e.re;
        a.iE[vb + a.G.ve(r)] = e.im;
      }
      if (a.info && lane == 0) a.info[m] = nfail;
      if (MODE != SC_FUSED || (a.flags & VEIG_WRITE_SCHUR))
        for (int c = 0; c < n; ++c)
          for (int r = lane; r < n; r += 64) {
            const int64_t idx = base + a.G.el(r, c);
            const cx<double> x = r <= c ? cldexp(ld<double>(t.at(r, c)), e2) : mk<double>(0, 0);
            a.rA[idx] = x.re;
            a.iA[idx] = x.im;
          }
    }
    if constexpr (MODE == SC_FUSED || MODE == SC_TREVC) {
      trevc_rows<P>(t, n, lane, top);
      __syncthreads();  // the eigenvector factor is ready
    }
  } else {
    // ---------------- the Schur vectors ----------------
    Rows z;
    z.init(lane);
    const int row0 = zi * Rows::RW, row = row0 + z.rl;
    bool rare = false;  // stages: an infinity or a NaN in the caller's matrix or rows
    if constexpr (MODE == SC_FUSED) {
      // the stages: the slots beside the one that the iteration is writing,
      // each as two vectors
      static_assert(schur_threads<SL, NT>() / 64 - 1 <= 2 * NT, "a stage for each wavefront");
      double2 *stage = &ring.step[1][0].c + zi * CAP;
      z.form_q(row, n, a.G, base, vb, a.rB, a.iB, a.rE, a.iE, stage);
    } else if constexpr (MODE == SC_ROOTS) {
#pragma unroll
      for (int c = 0; c < SL; ++c) z.z[c] = mk<double>(SL * z.h + c == row ? 1.0 : 0.0, 0);
    } else {
      z.load(row, n, a.G, base, a.rB, a.iB);
      rare = z.any_non_finite();
    }
    if constexpr (MODE == SC_LAHQR) {
      __syncthreads();  // the phases that made the subdiagonal real
#pragma unroll
      for (int c = 0; c < SL; ++c)
        if (SL * z.h + c < n) z.z[c] = mulc(z.z[c], ld<double>(&ring.step[1][0].c + SL * z.h + c));
    }
    if constexpr (MODE != SC_TREVC) z.start(ring, zi, zw);
    if constexpr (MODE == SC_LAHQR) rare = rare || __builtin_amdgcn_readfirstlane(ring.rare);
    if constexpr (MODE == SC_LAHQR || MODE == SC_TREVC) {
      if (__builtin_expect(rare, 0)) {  // the rest in the caller's planes
        if constexpr (MODE == SC_LAHQR) {
          z.store(row, n, a.G, base, a.rB, a.iB);
          __threadfence_block();  // a row's segments, to the lane that takes it
          replay_rare(&ring, lane < Rows::RW && row < n ? row : -1, a.G, base, a.rB, a.iB);
        } else {
          __syncthreads();  // the eigenvector factor is ready
          backtransform_rare<P>(t, row0, min(row0 + Rows::RW, n), n, lane, a.G, base, a.rB, a.iB);
        }
        return;
      }
    }
    if constexpr (MODE != SC_TREVC) z.replay(ring);
    if constexpr (MODE == SC_FUSED || MODE == SC_TREVC) {
      __syncthreads();  // the eigenvector factor is ready
      backtransform_mfma(t, z, row0, n, a.G, base, a.rB, a.iB);
    } else {
      z.store(row, n, a.G, base, a.rB, a.iB);
    }
  }
}

int set_lds(const void *kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    VEIG_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return VEIG_OK;
}

template <int CAP, int W, int MODE>
int launch_reduce(const BigArgs &a, hipStream_t s) {
  using S = ReduceBlock<CAP, W>;
  const size_t bytes = sizeof(S) + CAP * sizeof(double2);  // and tau
  VEIG_TRY(set_lds((const void *)k_reduce<CAP, W, MODE>, bytes));
  hipLaunchKernelGGL((k_reduce<CAP, W, MODE>), dim3((unsigned)a.G.nmat), dim3(S::kThreads), bytes, s, a);
  VEIG_HIP(hipGetLastError());
  return VEIG_OK;
}

template <int MODE>
int reduce_for(const BigArgs &a, hipStream_t s) {
  if (a.G.n <= 16) return launch_reduce<16, 4, MODE>(a, s);
  if (a.G.n <= 24) return launch_reduce<24, 2, MODE>(a, s);
  if (a.G.n <= 32) return launch_reduce<32, 4, MODE>(a, s);
  if (a.G.n <= 48) return launch_reduce<48, 4, MODE>(a, s);
  if (a.G.n <= 64) return launch_reduce<64, 4, MODE>(a, s);
  if (a.G.n <= 80) return launch_reduce<80, 8, MODE>(a, s);
  return launch_reduce<96, 6, MODE>(a, s);
}

template <int SL, int NT, int MODE>
int launch_schur(const BigArgs &a, hipStream_t s) {
  using Rows = SchurRows<SL, NT>;
  const size_t bytes =
      (MODE == SC_TREVC ? 0 : sizeof(typename Rows::Ring)) + (size_t)BandTile::entries(a.G.n) * sizeof(double2);
  const unsigned threads = 64u * (1 + (a.G.n + Rows::RW - 1) / Rows::RW);
  VEIG_TRY(set_lds((const void *)k_schur<SL, NT, MODE>, bytes));
  hipLaunchKernelGGL((k_schur<SL, NT, MODE>), dim3((unsigned)a.G.nmat), dim3(threads), bytes, s, a);
  VEIG_HIP(hipGetLastError());
  return VEIG_OK;
}

template <int MODE>
int schur_for(const BigArgs &a, hipStream_t s, int64_t batch) {
  if (a.G.n <= 32) return launch_schur<16, 2, MODE>(a, s);
  if (a.G.n <= 40) return launch_schur<20, 2, MODE>(a, s);
  if (a.G.n <= 48) return launch_schur<24, 2, MODE>(a, s);
  if (a.G.n <= 64) return launch_schur<32, 2, MODE>(a, s);
  // two matrices per CU at most: the shorter segments replay sooner (order 79 x
  // 64: 3.96 against 4.11 ms), past that the fewer wavefronts win
  if (a.G.n <= 80 && few_matrices(batch, 2)) return launch_schur<20, 4, MODE>(a, s);
  if (a.G.n <= 80) return launch_schur<40, 2, MODE>(a, s);
  // The stages load and store the rows of the caller, which 48 columns to a lane
  // spill (1.9 KB of scratch against 0.3 with 24): ztrevc always takes the shorter
  // segments (3,328 matrices, 48 -> 24 columns: order 81 4.01 -> 2.54 ms, 88 4.51 ->
  // 2.89, 93 4.71 -> 3.16), zlahqr up to four matrices per CU (1,024: order 81 8.74
  // -> 7.81 ms, 88 10.0 -> 9.1; 3,328: 28.6 -> 29.6, 32.7 -> 34.4) and where one
  // matrix per CU is all that fits (order 94 x 3,328 63.5 -> 60.8), not where their
  // longer ring is what leaves one (orders 90..93: 93 x 3,328 35.8 -> 59.5)
  if constexpr (MODE == SC_TREVC) return launch_schur<24, 4, MODE>(a, s);
  if constexpr (MODE == SC_LAHQR)
    if (a.G.n > 93 || (a.G.n < 90 && few_matrices(batch, 4))) return launch_schur<24, 4, MODE>(a, s);
  return launch_schur<48, 2, MODE>(a, s);
}

}  // namespace

namespace veig {

int launch_big(int mode, const Geom &G, double *rA, double *iA, double *rB, double *iB, double *rE, double *iE,
               int32_t *info, int itmax, uint32_t flags, hipStream_t s, const int32_t *list,
               const int32_t *list_count, const double *rC, const double *iC, int64_t batch) {
  if (G.n > VEIG_MAX_DIM) return fail(VEIG_ERR_UNSUPPORTED, "order beyond VEIG_MAX_DIM");
  if (G.nmat > INT32_MAX) return fail(VEIG_ERR_INVALID, "batch too large for one launch");
  const BigArgs a{rA, iA, rB, iB, rE, iE, info, G, itmax > 0 ? itmax : 30, flags, list, list_count, rC, iC};
  if (!batch) batch = G.nmat;
  switch (mode) {
    case BIG_FUSED:
      VEIG_TRY(reduce_for<RD_FUSED>(a, s));
      return schur_for<SC_FUSED>(a, s, batch);
    case BIG_REDUCE:  // orders 17..32
      return G.n <= 24 ? launch_reduce<24, 2, RD_BANDED>(a, s) : launch_reduce<32, 4, RD_BANDED>(a, s);
    case BIG_GEHRD: return reduce_for<RD_GEHRD>(a, s);
    case BIG_HESS: return reduce_for<RD_HESS>(a, s);
    case BIG_UNGHR: return reduce_for<RD_UNGHR>(a, s);
    case BIG_LAHQR: return schur_for<SC_LAHQR>(a, s, batch);
    case BIG_TREVC: return schur_for<SC_TREVC>(a, s, batch);
    default:  // BIG_ROOTS: orders up to VEIG_MAX_DIM_FAST
      return G.n <= 48 ? launch_schur<24, 2, SC_ROOTS>(a, s) : launch_schur<32, 2, SC_ROOTS>(a, s);
  }
}

}  // namespace veig
