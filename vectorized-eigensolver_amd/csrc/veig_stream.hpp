// One matrix per workgroup (orders 33..96, and lower ones in small batches): the pieces
// of the FP64 solve that the kernels of veig_big.hip, veig_roots.hip and
// veig_varsize.hip are made of.
//
//   reduce_block    the Hessenberg reduction on a dense LDS tile, every thread
//                   owning a chunk of one row (right update) or column (left);
//   lahqr_stream    the single-shift QR iteration by ONE wavefront, which
//                   records each sweep's rotations instead of applying them
//                   to the Schur vectors;
//   SchurRows       the Schur vectors in the registers of the other
//                   wavefronts, which replay the recorded sweeps, a few sweeps
//                   behind;
//   trevc_rows      the eigenvectors of the triangular factor.
//
// What bounds the QR iteration is the chain through the bulge: step K + 1
// needs two entries that step K has just rotated.  Exchanged through LDS, as
// the lane-group kernels do, a step is a store, a fence and two load round
// trips long (about 1,800 cycles at n = 64 on four wavefronts per SIMD).  So
// the 2 x 2 window of the chain lives in registers, computed alike by every
// lane; only the entry that the next column brings in crosses lanes, by
// readlane.  The rest of the matrix streams past it: lane t carries the
// running entry of column t (rows K, K+1 rotate) and of row t (columns K, K+1
// rotate), so each update is one load and one store per lane instead of two
// of each, and none of them is on the chain.
#pragma once
#include "veig_chain.hpp"
#include "veig_common.hpp"

namespace veig {

// The Hessenberg part, row <= col + 1, column c from c(c+3)/2, or a dense
// column-major tile.  Entries past the last are read (never used): kPad more
// are allocated, the last of them to be written where a lane has nothing to write.
struct BandTile {
  double2 *h;
  static constexpr int kPad = 2;
  __device__ __forceinline__ double2 *spare(int n) const { return h + entries(n) - 1; }
  static __host__ __device__ constexpr int entries(int n) { return ((n - 1) * (n + 2)) / 2 + n + kPad; }
  static __device__ __forceinline__ int off(int c) { return (c * (c + 3)) >> 1; }
  static __device__ __forceinline__ int width(int c) { return c + 2; }  // off(c + 1) - off(c)
  __device__ __forceinline__ double2 *at(int r, int c) const { return h + off(c) + r; }
};
template <int LD>
struct DenseTile {
  double2 *h;
  static __device__ __forceinline__ int off(int c) { return c * LD; }
  static __device__ __forceinline__ int width(int) { return LD; }
  __device__ __forceinline__ double2 *at(int r, int c) const { return h + off(c) + r; }
};

// keeps the compiler from moving LDS accesses across: one wavefront's LDS
// operations complete in order, so lanes need nothing more to see each other's
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ double read_lane(double x, int lane) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// The wavefront of the workgroup that runs the chain (chain_pick), the same in
// every wavefront.  ids: one LDS word per wavefront.  Every thread calls it (one
// barrier).
__device__ __forceinline__ int chain_wave(int *ids) {
  constexpr int kHwId = 4, kLdsAlloc = 6;  // hardware registers, read whole (32 bits from bit 0)
  const unsigned hw = __builtin_amdgcn_s_getreg((31 << 11) | kHwId);
  const unsigned lds = __builtin_amdgcn_s_getreg((31 << 11) | kLdsAlloc);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) ids[wave] = chain_note(wave, hw, lds);
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(chain_pick(ids, blockDim.x >> 6));
}

// sum over the wavefront, the same bits in every lane: rows of 16 by DPP, the
// four row sums by readlane
__device__ __forceinline__ double wave_sum(double x) {
  x = group_sum<16, double>(x);
  return (read_lane(x, 0) + read_lane(x, 16)) + (read_lane(x, 32) + read_lane(x, 48));
}

// the bits above the low word, without the sign: ordered as the magnitudes are,
// an infinity or a NaN from kNonFinite on
constexpr unsigned kNonFinite = 0x7ff00000u;
// the usual range of a largest entry: from 2^-300 to below 2^480
constexpr unsigned kUsualLow = (1023u - 300u) << 20, kUsualHigh = (1023u + 480u) << 20;
__device__ __forceinline__ unsigned high_word(double x) {
  return (unsigned)(__builtin_bit_cast(unsigned long long, x) >> 32) & 0x7fffffffu;
}
__device__ __forceinline__ unsigned high_word(cx<double> x) { return max(high_word(x.re), high_word(x.im)); }

// The power of two that a matrix is divided by before its squares are formed, 0
// where they fit as it is: with top (the largest high word) in the usual range the
// sums of its squares stay finite, and the square of an entry 2^-150 times the
// largest stays normal.  Exact, so the results are those of the unscaled matrix,
// scaled.
__device__ __forceinline__ int scale_exponent(unsigned top) {
  if ((top >= kUsualLow && top < kUsualHigh) || top >= kNonFinite) return 0;
  return (int)(top >> 20) - 1022;  // as frexp's (subnormal: -1022, small enough)
}
// a square below this is taken as zero: an entry below 2^-450, 2^-150 times the
// largest at most, whose square is on the way to losing its bits
constexpr double kTinySquare = 0x1p-900;

// count entries of a tile divided by 2^e, by `threads` threads
__device__ __forceinline__ void scale_entries(double2 *h, int count, int thread, int threads, int e) {
  for (int i = thread; i < count; i += threads) st<double>(h + i, cldexp(ld<double>(h + i), -e));
}

// The largest high word over the wavefront (exact where it is out of the usual
// range; in it, some lane's: two votes instead of six exchanges).
__device__ __forceinline__ unsigned wave_max(unsigned x) {
  if (__builtin_expect(__any(x >= kUsualLow) && !__any(x >= kUsualHigh), 1)) return kUsualLow;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = max(x, (unsigned)__shfl_xor((int)x, o));
  return (unsigned)__builtin_amdgcn_readfirstlane((int)x);
}

// the same over the wavefront's count entries
__device__ __forceinline__ unsigned wave_top(const double2 *h, int count, int lane) {
  unsigned x = 0;
  for (int i = lane; i < count; i += 64) x = max(x, high_word(ld<double>(h + i)));
  return wave_max(x);
}

// the same over the workgroup (one barrier; words: one LDS word per wavefront)
__device__ __forceinline__ unsigned block_max(unsigned x, unsigned *words) {
  x = wave_max(x);
  if ((threadIdx.x & 63) == 0) words[threadIdx.x >> 6] = x;
  __syncthreads();
  unsigned m = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) m = max(m, words[w]);
  return (unsigned)__builtin_amdgcn_readfirstlane((int)m);
}

// --------------------------------------------------------------------------
// The Hessenberg reduction (zgehrd, Toolbox.hpp:1315-1469, with zlarfg's
// LAPACK sign and its x = 0 guard) of the n x n matrix in a dense tile of
// capacity CAP, leaving the compact form: v(i+2:n) below the subdiagonal,
// tau(i) in tau_out (LDS, may be null).  Thread (r, q) owns the q-th of W chunks of row r (update
// from the right) and of column r (from the left): it takes its chunk and the
// reflector into registers, puts its partial product in LDS, and after a
// barrier adds the W partials in a fixed order and updates its chunk.  Every
// wavefront forms the reflector from column i (the same arithmetic on the same
// data).  Five barriers per reflector.  The tile is zero outside the matrix,
// so chunks need no bounds inside.
// kRare (the input holds an infinity or a NaN): a chunk's entries before the
// reflector's first are left out, not multiplied by the zeros of v, which would
// carry on what a finished row or column holds.  Entry by entry from LDS, and
// apart from the usual input's code: masks there cost order 64 x 65,536 180.4 ->
// 183.4 ms, the stages at order 40 x 2,048 3.09 -> 3.30.
// --------------------------------------------------------------------------
template <int CAP, int W>
struct ReduceBlock {
  static constexpr int LD = CAP | 1;  // odd: row-wise walks start on distinct banks
  static constexpr int CH = CAP / W;
  static constexpr int kThreads = (CAP * W + 63) / 64 * 64;
  static_assert(kThreads / 64 <= 12, "a word per wavefront");
  static_assert(LD == CAP + 1, "the reflector lives in the padding row");
  double2 H[LD * CAP];
  double2 part[W * CAP];
  unsigned words[12];  // block_max
  __device__ __forceinline__ double2 *at(int r, int c) { return H + c * LD + r; }
  __device__ __forceinline__ double2 *v(int c) { return H + c * LD + CAP; }  // the reflector's entry c
};

// kTiny: columns whose square is below kTinySquare are taken as zero (in a tile
// that has been scaled).
template <bool kRare, bool kTiny, int CAP, int W>
__device__ __forceinline__ void reduce_steps(ReduceBlock<CAP, W> &sm, int n, double2 *tau_out) {
  using R = double;
  constexpr int CH = ReduceBlock<CAP, W>::CH;
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = tid % CAP, q = tid / CAP, c0 = q * CH;
  const bool in = r < n && q < W;
  for (int i = 0; i + 1 < n; ++i) {
    // ---- reflector annihilating H(i+2:n, i) ----
    R part = 0.0;
    for (int k = lane; k < n; k += 64)
      if (k >= i + 2) part += abs2(ld<R>(sm.at(k, i)));
    const R xnorm2 = wave_sum(part);
    const cx<R> alpha = ld<R>(sm.at(i + 1, i));
    cx<R> tau = mk<R>(0, 0), scal = mk<R>(0, 0);
    R beta = alpha.re;
    const R nrm2 = abs2(alpha) + xnorm2;
    if (!(xnorm2 == 0.0 && alpha.im == 0.0) && !(kTiny && nrm2 < kTinySquare)) {
      const R nrm = fsqrt(nrm2);
      beta = alpha.re >= 0.0 ? -nrm : nrm;
      const R ib = frcp(beta);
      tau = mk((beta - alpha.re) * ib, -alpha.im * ib);
      scal = inv(mk(alpha.re - beta, alpha.im));
    }
    cx<R> vr = mk<R>(0, 0);
    if (q == 0) {
      if (r == i + 1) vr = mk<R>(1, 0);
      else if (r >= i + 2 && in) vr = mul(ld<R>(sm.at(r, i)), scal);
      st<R>(sm.v(r), vr);
    }
    if (tau_out && tid == 0) st<R>(tau_out + i, tau);
    __syncthreads();
    const bool mine = in && c0 + CH - 1 > i && c0 < n;
    const int cr = c0 > i ? c0 : i + 1, ce = min(c0 + CH, n);  // kRare: these of the chunk
    // ---- H <- H (I - tau v v^H): row r, columns of the chunk ----
    cx<R> h[CH], v[CH];
    cx<R> w = mk<R>(0, 0);
    if (mine) {
      if constexpr (kRare) {
#pragma unroll 1
        for (int c = cr; c < ce; ++c) w = add(w, mul(ld<R>(sm.at(r, c)), ld<R>(sm.v(c))));
      } else {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
          h[j] = ld<R>(sm.at(r, c0 + j));
          v[j] = ld<R>(sm.v(c0 + j));  // zero at c <= i and beyond n
        }
#pragma unroll
        for (int j = 0; j < CH; ++j) w = add(w, mul(h[j], v[j]));
      }
    }
    if (q < W) st<R>(sm.part + q * CAP + r, w);
    __syncthreads();
    if (q == 0 && in && r >= i + 1) st<R>(sm.at(r, i), r == i + 1 ? mk<R>(beta, 0.0) : vr);
    if (mine) {
      w = mk<R>(0, 0);
#pragma unroll
      for (int p = 0; p < W; ++p) w = add(w, ld<R>(sm.part + p * CAP + r));
      w = mul(tau, w);
      if constexpr (kRare) {
#pragma unroll 1
        for (int c = cr; c < ce; ++c) st<R>(sm.at(r, c), sub(ld<R>(sm.at(r, c)), mulc(w, ld<R>(sm.v(c)))));
      } else {
#pragma unroll
        for (int j = 0; j < CH; ++j)
          if (c0 + j > i) st<R>(sm.at(r, c0 + j), sub(h[j], mulc(w, v[j])));
      }
    }
    __syncthreads();
    // ---- H <- (I - conj(tau) v v^H) H: column r > i, rows of the chunk ----
    const bool left = mine && r > i;
    cx<R> y = mk<R>(0, 0);
    if (left) {
      if constexpr (kRare) {
#pragma unroll 1
        for (int c = cr; c < ce; ++c) y = add(y, cmul(ld<R>(sm.v(c)), ld<R>(sm.at(c, r))));
      } else {
#pragma unroll
        for (int j = 0; j < CH; ++j) h[j] = ld<R>(sm.at(c0 + j, r));
#pragma unroll
        for (int j = 0; j < CH; ++j) y = add(y, cmul(v[j], h[j]));
      }
    }
    if (q < W) st<R>(sm.part + q * CAP + r, y);
    __syncthreads();
    if (left) {
      y = mk<R>(0, 0);
#pragma unroll
      for (int p = 0; p < W; ++p) y = add(y, ld<R>(sm.part + p * CAP + r));
      y = cmul(tau, y);  // conj(tau) * y
      if constexpr (kRare) {
#pragma unroll 1
        for (int c = cr; c < ce; ++c) st<R>(sm.at(c, r), sub(ld<R>(sm.at(c, r)), mul(ld<R>(sm.v(c)), y)));
      } else {
#pragma unroll
        for (int j = 0; j < CH; ++j)
          if (c0 + j > i) st<R>(sm.at(c0 + j, r), sub(h[j], mul(v[j], y)));
      }
    }
    __syncthreads();
  }
}

template <int CAP, int W>
__device__ __forceinline__ void scale_tile(ReduceBlock<CAP, W> &sm, int e) {
  scale_entries(sm.H, (int)(sizeof(sm.H) / sizeof(double2)), threadIdx.x, blockDim.x, e);
  __syncthreads();
}
// the rare forms as calls: inlined, they cost the usual input's kernels 1 to 3% at
// the capacities from 48 on, in registers and in the order that the rest came out in
template <int CAP, int W>
__device__ __noinline__ void scale_call(ReduceBlock<CAP, W> *sm, int e) {
  scale_tile(*sm, e);
}
template <bool kScale, int CAP, int W>
__device__ __noinline__ void reduce_call(ReduceBlock<CAP, W> *sm, int n, double2 *tau_out) {
  reduce_steps<true, kScale>(*sm, n, tau_out);
}

// top: the largest high word of the input, from reduce_load.  Returns the e of
// the 2^e that the tile's H is divided by (scale_exponent).  (Calls cost a launch
// about a microsecond, so not at the capacities that small batches take: zgehrd of
// 64 matrices of order 8 14.6 us with them, 13.7 without.)
// kScale = false, for the QR iteration on lane groups, which does not scale: a
// matrix out of the range stays undefined, as there, where its H would come out of
// an iteration without squares as converged and wrong.
template <bool kScale, int CAP, int W>
__device__ __forceinline__ int reduce_block(ReduceBlock<CAP, W> &sm, int n, unsigned top, double2 *tau_out) {
  constexpr bool kCall = CAP > 32;
  const int e = kScale ? scale_exponent(top) : 0;
  if (__builtin_expect(e != 0, 0)) {
    if constexpr (kCall) scale_call(&sm, e);
    else scale_tile(sm, e);
  }
  if (__builtin_expect(top >= kNonFinite, 0)) {
    if constexpr (kCall) reduce_call<kScale>(&sm, n, tau_out);
    else reduce_steps<true, kScale>(sm, n, tau_out);
  } else {
    reduce_steps<false, kScale>(sm, n, tau_out);
  }
  return e;
}

// the tile from memory, zeros outside the matrix (ends at a barrier); returns the
// largest high word (block_max).  beside: what else is to be done before the
// barrier; returns the high word of what it loads.
template <int CAP, int W, typename F>
__device__ __forceinline__ unsigned reduce_load(ReduceBlock<CAP, W> &sm, int n, const Geom &G, int64_t base,
                                                const double *re, const double *im, F &&beside) {
  constexpr int CH = ReduceBlock<CAP, W>::CH;
  const int r = threadIdx.x % CAP, q = threadIdx.x / CAP;
  unsigned top = 0;
  if (q < W) {
    cx<double> x[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int c = q * CH + j;
      x[j] = mk<double>(0, 0);
      if (r < n && c < n) {
        const int64_t idx = base + G.el(r, c);
        x[j] = mk<double>(re[idx], im[idx]);
      }
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      top = max(top, high_word(x[j]));
      st<double>(sm.at(r, q * CH + j), x[j]);
    }
  }
  return block_max(max(top, beside()), sm.words);
}

// the tile to memory, H times 2^e (the reflectors below its subdiagonal as they are)
template <int CAP, int W>
__device__ __forceinline__ void reduce_store(ReduceBlock<CAP, W> &sm, int n, const Geom &G, int64_t base, double *re,
                                             double *im, int e) {
  constexpr int CH = ReduceBlock<CAP, W>::CH;
  const int r = threadIdx.x % CAP, q = threadIdx.x / CAP;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int c = q * CH + j;
    if (q < W && r < n && c < n) {
      const int64_t idx = base + G.el(r, c);
      const cx<double> x = cldexp(ld<double>(sm.at(r, c)), r <= c + 1 ? e : 0);
      re[idx] = x.re;
      im[idx] = x.im;
    }
  }
}

// Q = H_0 H_1 ... H_{n-2} (zunghr, Toolbox.hpp:1470-1659) from the compact
// form in the tile, thread (r, q) holding its chunk of row r in registers; two
// barriers per reflector, before and after the partial sums are read
template <int CAP, int W>
__device__ __forceinline__ void form_q_block(ReduceBlock<CAP, W> &sm, int n, const double2 *tau_in,
                                             cx<double> (&z)[ReduceBlock<CAP, W>::CH]) {
  using R = double;
  constexpr int CH = ReduceBlock<CAP, W>::CH;
  const int r = threadIdx.x % CAP, q = threadIdx.x / CAP, c0 = q * CH;
#pragma unroll
  for (int j = 0; j < CH; ++j) z[j] = mk<R>(c0 + j == r ? 1.0 : 0.0, 0.0);
  for (int i = 0; i + 1 < n; ++i) {
    const cx<R> tau = ld<R>(tau_in + i);
    const bool mine = q < W && c0 + CH - 1 > i && c0 < n;
    cx<R> v[CH];
    cx<R> w = mk<R>(0, 0);
    if (mine) {
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int c = c0 + j;
        v[j] = ld<R>(sm.at(c, i));  // zero beyond n
        if (c <= i + 1) v[j] = mk<R>(c == i + 1 ? 1.0 : 0.0, 0.0);
      }
#pragma unroll
      for (int j = 0; j < CH; ++j) w = add(w, mul(z[j], v[j]));
    }
    if (q < W) st<R>(sm.part + q * CAP + r, w);
    __syncthreads();
    if (mine) {
      w = mk<R>(0, 0);
#pragma unroll
      for (int p = 0; p < W; ++p) w = add(w, ld<R>(sm.part + p * CAP + r));
      w = mul(tau, w);
#pragma unroll
      for (int j = 0; j < CH; ++j) z[j] = sub(z[j], mulc(w, v[j]));
    }
    __syncthreads();
  }
}

// form_q_block for an input that holds an infinity or a NaN (see reduce_block):
// a reflector leaves the columns before its first alone.  The chunk is kept in
// the output planes, each thread using its own entries only.
template <int CAP, int W>
__device__ __forceinline__ void form_q_rare(ReduceBlock<CAP, W> &sm, int n, const double2 *tau_in, const Geom &G,
                                            int64_t base, double *re, double *im) {
  using R = double;
  constexpr int CH = ReduceBlock<CAP, W>::CH;
  const int r = threadIdx.x % CAP, q = threadIdx.x / CAP, c0 = q * CH;
  const int end = q < W && r < n ? min(c0 + CH, n) : 0;
  auto get = [&](int c) { return mk<R>(re[base + G.el(r, c)], im[base + G.el(r, c)]); };
  auto put = [&](int c, cx<R> x) {
    re[base + G.el(r, c)] = x.re;
    im[base + G.el(r, c)] = x.im;
  };
  for (int c = c0; c < end; ++c) put(c, mk<R>(c == r ? 1.0 : 0.0, 0.0));
  for (int i = 0; i + 1 < n; ++i) {
    const int cr = c0 > i ? c0 : i + 1;
    auto v = [&](int c) { return c == i + 1 ? mk<R>(1, 0) : ld<R>(sm.at(c, i)); };
    cx<R> w = mk<R>(0, 0);
#pragma unroll 1
    for (int c = cr; c < end; ++c) w = add(w, mul(get(c), v(c)));
    if (q < W) st<R>(sm.part + q * CAP + r, w);
    __syncthreads();
    w = mk<R>(0, 0);
    if (q < W)
      for (int p = 0; p < W; ++p) w = add(w, ld<R>(sm.part + p * CAP + r));
    w = mul(ld<R>(tau_in + i), w);
#pragma unroll 1
    for (int c = cr; c < end; ++c) put(c, sub(get(c), mulc(w, v(c))));
    __syncthreads();
  }
}

// --------------------------------------------------------------------------
// records of the sweeps
// --------------------------------------------------------------------------
// A ring of R sweeps of rotations for steps 0..CAP-1; a step outside its
// sweep holds the identity, so the Schur-vector wavefronts apply every entry
// without asking.  Entry K: (Re c, Im c) and (s, r^2), r the step's new H(K, K-1)
// (the iteration's own use).
struct StepRec {
  double2 c, sr;
};
template <int CAP_, int R_>
struct SweepRing {
  static constexpr int CAP = CAP_, R = R_;
  static constexpr bool kReplayed = true;
  StepRec step[R][CAP];
  double2 ph[R];   // conj(h/|h|) of the sweep's last step: column I is scaled by its conjugate
  int L[R], I[R];  // steps L..I-1
  int last[R];
  int simd[8];     // chain_wave
  int rare;        // the Hessenberg matrix holds an infinity or a NaN
};
// the record of a wavefront that keeps no Schur vectors: this sweep's r^2 only
template <int CAP_>
struct SweepScratch {
  static constexpr int CAP = CAP_, R = 1;
  static constexpr bool kReplayed = false;
  StepRec step[1][CAP];
  int simd[4];
};

template <int CAP, int R>
__device__ __forceinline__ void ring_identity(SweepRing<CAP, R> &ring, int slot, int lane, int last) {
  for (int t = lane; t < CAP; t += 64) ring.step[slot][t] = StepRec{double2{1.0, 0.0}, double2{0.0, 0.0}};
  if (lane == 0) {
    ring.L[slot] = ring.I[slot] = 0;  // no steps; column 0 is never scaled
    ring.last[slot] = last;
  }
}

// --------------------------------------------------------------------------
// the Wilkinson shift (see lahqr): h11 h12 / h21 h22 the trailing 2 x 2 block.
// Its root and reciprocal are good to 2^-47.8, here as in lahqr: it steers the
// iteration and does not enter the similarity.  Measured with both to the last
// bit, against extended precision (orders 33..96, Gaussian, Hermitian and cond(V)
// = 1e3): backward error 3.1e-16 in the mean either way, the eigenvalues' error
// 5e-16 to 9e-16 of the norm either way (the reflectors' kernels that these
// replaced at 33..64: 2.6e-16 to 6.6e-16, 7e-16 to 1.7e-15).
// --------------------------------------------------------------------------
__device__ __forceinline__ cx<double> wilkinson_shift(cx<double> h11, cx<double> h12, cx<double> h21,
                                                      cx<double> h22) {
  using R = double;
  const cx<R> u2 = mul(h12, h21);
  if (u2.re == 0.0 && u2.im == 0.0) return h22;
  const cx<R> x = scale(sub(h11, h22), 0.5);
  const R sx = cabs1(x);
  const int eu = fexp(cabs1(u2)), ex = sx > 0.0 ? fexp(sx) : -4096;
  const int E = max((eu + 1) >> 1, ex);
  const cx<R> xs = cldexp(x, -E);
  cx<R> ys = csqrt_unit(add(mul(xs, xs), cldexp(u2, -2 * E)));
  if (sx > 0.0 && xs.re * ys.re + xs.im * ys.im < 0.0) ys = mk(-ys.re, -ys.im);
  const cx<R> d = add(xs, ys);
  const R id = frcp1(abs2(d));
  return sub(h22, mul(cldexp(u2, -E), mk(d.re * id, -d.im * id)));
}

// the subdiagonal made real (loop 20 of zlahqr_schur, Toolbox.hpp:735-793),
// by one wavefront; the scaling of Schur-vector column i goes to ph[i]
// (z_i <- z_i conj(ph[i])), 1 where there is none
template <typename T>
__device__ __forceinline__ void make_subdiag_real(const T &t, int n, int lane, double2 *ph) {
  using R = double;
  for (int i = lane; i < n; i += 64) ph[i] = double2{1.0, 0.0};
  lds_order();
  for (int i = 1; i < n; ++i) {
    const cx<R> h = ld<R>(t.at(i, i - 1));
    lds_order();
    if (h.im != 0.0) {  // uniform: every lane reads the same entry
      const cx<R> w = scale(h, frcp(cabs1(h)));
      const cx<R> sc = scale(conj(w), frsq(abs2(w)));  // conj(h/|h|)
      if (lane == 0) {
        st<R>(t.at(i, i - 1), mk(fsqrt(abs2(h)), 0.0));
        st<R>(ph + i, sc);
      }
      for (int x = i + lane; x < n; x += 64) st<R>(t.at(i, x), mul(ld<R>(t.at(i, x)), sc));
      lds_order();
      for (int x = lane; x <= i + 1 && x < n; x += 64) st<R>(t.at(x, i), mulc(ld<R>(t.at(x, i)), sc));
      lds_order();
    }
  }
}

// --------------------------------------------------------------------------
// the QR iteration (zlahqr_schur, Toolbox.hpp:690-1031; TZ = false: the
// eigenvalues-only zlahqr_, 1663-1890, which touches the active block only)
// by one wavefront, lane t owning row and column t (and t + 64: P = 2).
// Deflation test, shifts and iteration cap as lahqr's.  RING: a SweepRing,
// published at one workgroup barrier per sweep (and drained at the end by as
// many as the ring is deep), or NoRing.  Returns the eigenvalues accepted at
// the iteration cap.
//
// A wavefront alone issues one instruction per 5 cycles, so the step's
// instruction count is its time: the 51 FP64 instructions it cannot do without
// (the rotation 12, the window 27, the update of rows and columns 12) and as
// few others as possible.  Hence: one update for the lanes ahead of the bulge
// and behind it, stores without execution masks (lanes past the order repeat
// the last column), record entries written by every lane, running addresses.
// --------------------------------------------------------------------------
struct StreamWindow {
  cx<double> a0;   // H(K, K-1): the rotation's input
  double a1;       // H(K+1, K-1), real
  double m2;       // |a0|^2 + a1^2
  cx<double> x1;   // H(K, K)
  cx<double> x2;   // H(K+1, K)
  double hs;       // H(K+2, K+1), real, not yet rotated
  uint64_t none, none_hi;  // bit K (K - 64): step K's input was zero, its rotation the identity
  cx<double> was;       // a0 where the last one was replaced

  // m2, and the zero vector (or one below kTinySquare) replaced
  // by one that gives G = I
  __device__ __forceinline__ void norm(int K) {
    m2 = fma(a0.re, a0.re, fma(a0.im, a0.im, a1 * a1));
    if (__builtin_expect(__any(m2 < kTinySquare), 0)) {
      was = a0;
      a0 = mk<double>(1, 0);
      a1 = 0.0;
      m2 = 1.0;
      const uint64_t bit = 1ull << (K & 63);
      none |= K < 64 ? bit : 0;
      none_hi |= K < 64 ? 0 : bit;
    }
  }
};

// The running state of a sweep.  Lane t is ahead of the bulge (t > K) or behind
// it (t < K), and the two updates it then takes part in are the same one but
// for the sign of Im c (rot_left by q is rot_right by its conjugate): ahead,
// rows K, K+1 of column t by this step's rotation; behind, columns K-1, K of
// row t by the last one's (these lag by a step, so that row K has its entry
// of column K+1).  So one update serves both, 12 FP64 instructions and one
// store and load per lane, and a lane changes its role as the bulge passes it.
// (Each lane taking both updates at every step, half of them to no use: order
// 64 x 65,536 198 ms instead of 181.  All lanes a step behind the
// window, so that the update fills the latency of the reciprocal square root:
// 191 ms, the window then having an entry more to rotate.)
template <int P>
struct StreamLanes {
  cx<double> e[P];     // the running entry: H(K, t) ahead, H(t, K-1) behind
  cx<double> o[P];     // the entry that the next rotation pairs it with
  Rot<double> q;       // the last step's rotation
  double sd[P];        // H(t + 2, t + 1), real
  double2 *pe[P], *po[P];  // their places in the tile
  int t[P];            // this lane's row and column
};

// step K; M: the slot that the bulge is passing (slots before it are behind,
// slots after it ahead), Y: the slot of column K + 1; REC: the whole record,
// or r^2 only
template <int P, int M, int Y, bool REC, typename T>
__device__ __forceinline__ void stream_step(int K, StreamWindow &x, StreamLanes<P> &a, StepRec *rec) {
  using R = double;
  const R m2 = x.m2, ir = frsq(m2);
  const Rot<R> q{mk(x.a0.re * ir, x.a0.im * ir), x.a1 * ir};
  if constexpr (REC) {
    rec[K].c = double2{q.c.re, q.c.im};
    rec[K].sr = double2{q.s, m2};
  } else {
    rec[K].sr.y = m2;
  }
  const int wk = T::width(K);
  bool ahead[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    ahead[p] = p > M || (p == M && a.t[p] > K);
    const Rot<R> g{mk(ahead[p] ? q.c.re : a.q.c.re, ahead[p] ? -q.c.im : a.q.c.im), ahead[p] ? q.s : a.q.s};
    cx<R> out = a.e[p];
    rot_right(g, out, a.o[p]);
    a.e[p] = a.o[p];
    st<R>(a.pe[p], out);  // (lane K: overwritten by itself at the next step)
  }
  // the window: column K of rows K, K+1, then row K+1 of columns K, K+1
  cx<R> x1 = x.x1, x2 = x.x2;
  rot_left(q, x1, x2);
  const int src = (K + 1) & 63;
  cx<R> y2 = mk(read_lane(a.e[Y].re, src), read_lane(a.e[Y].im, src));
  rot_right(q, x2, y2);
  x.a0 = x2;
  x.x1 = y2;
  x.a1 = q.s * x.hs;
  x.norm(K + 1);
  x.x2 = mk(q.c.re * x.hs, -q.c.im * x.hs);
  x.hs = read_lane(a.sd[Y], src);
  a.q = q;
  lds_order();
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const bool pass = p == M && a.t[p] == K;  // the bulge passes lane K: x1 is row K's first entry
    a.e[p] = mk(pass ? x1.re : a.e[p].re, pass ? x1.im : a.e[p].im);
    a.pe[p] = pass ? a.pe[p] : a.po[p];
    a.po[p] = a.pe[p] + (ahead[p] ? 1 : wk);
    a.o[p] = ld<R>(a.po[p]);  // past the last row and column: read and not used
  }
}

template <int P, bool TZ, typename T, typename RING>
__device__ __forceinline__ int lahqr_stream(const T &t, int n, int lane, RING &ring, int itmax) {
  using R = double;
  constexpr bool kRec = RING::kReplayed;
  constexpr int CAP = RING::CAP, kR = RING::R;
  static_assert(TZ || P == 1, "the active block's lanes sit in one slot");
  const R ulp = limits<R>::eps;
  const R smlnum = limits<R>::tiny * (R(n > 0 ? n : 1) / ulp);
  int rt[P];  // lanes past the order repeat its last row and column
#pragma unroll
  for (int p = 0; p < P; ++p) rt[p] = lane + 64 * p < n ? lane + 64 * p : n - 1;
  int I = n - 1, L = 0, its = 0, nfail = 0, slot = 0;
  bool first = true;  // kRec: the other wavefronts are still forming Q
  while (I >= 0) {
    if (its > itmax) {  // accepted without convergence (the reference's silent case)
      ++nfail;
      --I;
      its = 0;
      continue;
    }
    // ---- deflation: every subdiagonal entry k = 1..I at once ----
    uint64_t neg[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int k = lane + 64 * p;
      bool ng = false;
      if (k > 0 && k <= I) {
        const cx<R> h = ld<R>(t.at(k, k - 1)), hkk1 = ld<R>(t.at(k - 1, k - 1)), hkk = ld<R>(t.at(k, k));
        R tst = cabs1(hkk1) + cabs1(hkk);
        if (__builtin_expect(__any(tst == 0.0), 0)) {
          if (tst == 0.0) {
            if (k - 2 >= 0) tst += fabs(t.at(k - 1, k - 2)->x);
            if (k + 1 <= n - 1) tst += fabs(t.at(k + 1, k)->x);
          }
        }
        ng = cabs1(h) <= smlnum;
        if (!ng && fabs(h.re) <= ulp * tst) {
          const cx<R> hup = ld<R>(t.at(k - 1, k));
          const R ab = fmax(cabs1(h), cabs1(hup)), ba = fmin(cabs1(h), cabs1(hup));
          const R d3 = cabs1(sub(hkk1, hkk));
          const R aa = fmax(cabs1(hkk), d3), bb = fmin(cabs1(hkk), d3);
          const R s = aa + ab;  // >= cabs1(h) > 0
          if constexpr (TZ) {
            ng = ba * (ab / s) <= fmax(smlnum, ulp * (bb * (aa / s)));  // (s may be infinite)
          } else {
            const R is = frcp(s);
            ng = ba * (ab * is) <= fmax(smlnum, ulp * (bb * (aa * is)));
          }
        }
      }
      neg[p] = __ballot(ng);
    }
    lds_order();
    for (;;) {
      L = 0;  // the highest negligible k <= I
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int top = I - 64 * p;  // bits 0..top of this word
        const uint64_t c = top < 0 ? 0 : (top >= 63 ? neg[p] : neg[p] & ((2ull << top) - 1));
        if (c) L = 64 * p + 63 - __clzll(c);
      }
      if (L > 0 && lane == 0) st<R>(t.at(L, L - 1), mk<R>(0, 0));
      if (L < I) break;
      --I;  // H(I, I) has deflated
      its = 0;
      if (I < 0) break;
    }
    lds_order();
    if (I < 0) break;

    // ---- shift and first column (Toolbox.hpp:896-1015) ----
    const cx<R> h11 = ld<R>(t.at(L, L));
    const R h21 = t.at(L + 1, L)->x;
    cx<R> sh;
    if (__builtin_expect(its == 10, 0)) {
      sh = h11;
      sh.re += 0.75 * fabs(h21);
    } else if (__builtin_expect(its == 20, 0)) {
      sh = ld<R>(t.at(I, I));
      sh.re += 0.75 * fabs(t.at(I, I - 1)->x);
    } else {
      sh = wilkinson_shift(ld<R>(t.at(I - 1, I - 1)), ld<R>(t.at(I - 1, I)), ld<R>(t.at(I, I - 1)),
                           ld<R>(t.at(I, I)));
    }
    const cx<R> h11s = sub(h11, sh);
    const int E1 = fexp(cabs1(h11s) + fabs(h21));
    StreamWindow x;
    x.a0 = cldexp(h11s, -E1);
    x.a1 = fldexp(h21, -E1);
    x.none = x.none_hi = 0;
    x.norm(L);
    x.x1 = h11;
    x.x2 = mk<R>(h21, 0.0);
    x.hs = t.at(L + 2, L + 1)->x;  // past the last row: read and not used

    // ---- the sweep (Toolbox.hpp:138-335) ----
    // the identity as the rotation before the first, of (0, H(t, L)), brings
    // column L into the row updates (of what is above the active block: column
    // L - 1 may hold an infinity that column L does not, and the other way round)
    StreamLanes<P> a;
    a.q = Rot<R>{mk<R>(1, 0), 0.0};
    StepRec *rec = ring.step[slot];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      // lanes past the order repeat the last column, always ahead; without
      // the Schur form the lanes outside the active block repeat column I
      const int t0 = lane + 64 * p;
      const bool in = TZ || (t0 >= L && t0 <= I);
      const int at = in ? rt[p] : I;
      a.t[p] = in ? t0 : I;
      const bool behind = a.t[p] < L;
      a.po[p] = behind ? t.at(at, L) : t.at(L, at) + 1;
      a.pe[p] = a.po[p] - 1;
      a.e[p] = ld<R>(a.pe[p]);
      a.o[p] = ld<R>(a.po[p]);
      if constexpr (TZ) {
        if (behind) {
          a.pe[p] = t.spare(n);
          a.e[p] = mk<R>(0, 0);
        }
      }
      const int sc = t0 + 1 < I ? t0 + 1 : I - 1;
      a.sd[p] = t.at(sc + 1, sc)->x;
    }
    if constexpr (kRec) {
      for (int k = lane; k < CAP; k += 64)
        if (k < L || k >= I) rec[k] = StepRec{double2{1.0, 0.0}, double2{0.0, 0.0}};
    }
    // (two steps per turn: the state alternates between two sets of registers
    // instead of being copied)
    int K = L;
    auto run = [&](auto mc, auto yc, int end) {
      constexpr int M = decltype(mc)::value, Y = decltype(yc)::value;
      for (; K + 1 < end; K += 2) {
        stream_step<P, M, Y, kRec, T>(K, x, a, rec);
        stream_step<P, M, Y, kRec, T>(K + 1, x, a, rec);
      }
      if (K < end) {
        stream_step<P, M, Y, kRec, T>(K, x, a, rec);
        ++K;
      }
    };
    constexpr std::integral_constant<int, 0> s0;
    constexpr std::integral_constant<int, P - 1> s1;
    if constexpr (P == 1) {
      run(s0, s0, I);
    } else {
      // column K + 1 in the first slot, then row K (K = 63) in the first slot
      run(s0, s0, I < 63 ? I : 63);
      if (K == 63 && I > 63) {
        stream_step<P, 0, P - 1, kRec, T>(K, x, a, rec);
        ++K;
      }
      if (K < I) run(s1, s1, I);
    }
    // the last rotation's rows, then H(I, I-1) made real (Toolbox.hpp:337-367)
    // on the way out: row I right of I and column I above it scaled
    cx<R> zz = mk<R>(1, 0);
    cx<R> hsub = ((I < 64 ? x.none : x.none_hi) >> (I & 63)) & 1u ? x.was : x.a0;
    if (hsub.im != 0.0 && abs2(hsub) > kTinySquare) {  // a smaller h: negligible, or its real part is taken
      const R m2 = abs2(hsub), id = frsq(m2);
      zz = mk(hsub.re * id, -hsub.im * id);  // conj(h/|h|)
      hsub = mk(m2 * id, 0.0);
    }
    lds_order();
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int q = lane + 64 * p;
      cx<R> o = a.e[p], c = a.o[p];
      rot_right(a.q, o, c);
      if (q < I && (TZ || q >= L)) {
        st<R>(t.at(rt[p], I - 1), o);
        st<R>(t.at(rt[p], I), mulc(c, zz));
      }
      if (TZ && q > I && q < n) st<R>(t.at(I, rt[p]), mul(a.e[p], zz));
      if (q > L && q < I) {  // H(q, q-1) = r
        const R m2 = rec[q].sr.y, r = m2 * frsq(m2);
        st<R>(t.at(q, q - 1), mk<R>(((p == 0 ? x.none : x.none_hi) >> lane) & 1u ? 0.0 : r, 0.0));
      }
    }
    if (lane == 0) {
      st<R>(t.at(I, I - 1), hsub);
      st<R>(t.at(I, I), x.x1);
    }
    lds_order();
    ++its;
    if constexpr (kRec) {
      if (lane == 0) {
        st<R>(&ring.ph[slot], zz);
        ring.L[slot] = L;
        ring.I[slot] = I;
        ring.last[slot] = 0;
      }
      if (first) __syncthreads();  // the ring's other slots are free (SchurRows::start)
      first = false;
      __syncthreads();  // the sweep's record is out
      slot = slot + 1 == kR ? 0 : slot + 1;
    }
  }
  if constexpr (kRec) {
    if (first) __syncthreads();
    for (int d = 0; d + 2 < kR; ++d) {  // until the last segment has replayed the last sweep
      ring_identity(ring, slot, lane, d + 3 == kR);
      __syncthreads();
      slot = slot + 1 == kR ? 0 : slot + 1;
    }
  }
  return nfail;
}

// --------------------------------------------------------------------------
// The Schur vectors: NT lanes per row, lane segment h holding columns
// SL h .. SL h + SL - 1 of its row in registers; RW = 64 / NT rows per
// wavefront.  A sweep's rotations act on consecutive column pairs, so segment
// h replays its part of a sweep one sweep behind segment h - 1: every lane has
// a rotation at (almost) every step, where one sweep alone would keep one
// segment in NT busy.  The pair across a segment border is exchanged between
// the two lanes once per sweep, between the two segments' parts.
// --------------------------------------------------------------------------
template <int SL, int NT>
struct SchurRows {
  static constexpr int CAP = SL * NT;
  static constexpr int RW = 64 / NT;
  static constexpr int R = NT + 1;  // NT sweeps being replayed, one being recorded
  using Ring = SweepRing<CAP, R>;
  cx<double> z[SL];
  int lane, h, rl;  // segment, row within the wavefront

  __device__ __forceinline__ void init(int lane_) {
    lane = lane_;
    h = lane / RW;
    rl = lane % RW;
  }
  // the value of the same row's lane `d` segments up (d < 0: down)
  __device__ __forceinline__ cx<double> seg_shift(cx<double> x, int d) const {
    const int src = (lane + d * RW) & 63;
    return mk<double>(__shfl(x.re, src), __shfl(x.im, src));
  }
  __device__ __forceinline__ cx<double> row_sum(cx<double> x) const {
#pragma unroll
    for (int o = RW; o < 64; o <<= 1) x = add(x, mk<double>(__shfl_xor(x.re, o), __shfl_xor(x.im, o)));
    return x;
  }

  // Q = H_0 H_1 ... H_{n-2} (zunghr, Toolbox.hpp:1470-1659) from the compact
  // form's reflectors in the V and E planes: the wavefront stages v(i) in
  // LDS (stage: n entries of its own) and every lane applies it to its row
  __device__ __forceinline__ void form_q(int row, int n, const Geom &G, int64_t base, int64_t vbase, const double *rV,
                                         const double *iV, const double *rE, const double *iE, double2 *stage) {
#pragma unroll
    for (int c = 0; c < SL; ++c) z[c] = mk<double>(SL * h + c == row ? 1.0 : 0.0, 0);
    constexpr int P = (CAP + 63) / 64;
    cx<double> vn[P], tn;
    auto fetch = [&](int i) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int r = lane + 64 * p;
        vn[p] = mk<double>(r == i + 1 ? 1.0 : 0.0, 0);
        if (r >= i + 2 && r < n) {
          const int64_t idx = base + G.el(r, i);
          vn[p] = mk<double>(rV[idx], iV[idx]);
        }
      }
      tn = mk<double>(rE[vbase + G.ve(i)], iE[vbase + G.ve(i)]);
    };
    if (n > 1) fetch(0);
    for (int i = 0; i + 1 < n; ++i) {
      const cx<double> tau = tn;
#pragma unroll
      for (int p = 0; p < P; ++p)
        if (lane + 64 * p < CAP) st<double>(stage + lane + 64 * p, vn[p]);
      if (i + 2 < n) fetch(i + 1);
      lds_order();
      const double2 *vs = stage + SL * h;
      cx<double> wv = mk<double>(0, 0);
#pragma unroll
      for (int c = 0; c < SL; ++c) wv = add(wv, mul(z[c], ld<double>(vs + c)));
      const cx<double> tw = mul(tau, row_sum(wv));
      lds_order();  // read v again rather than keep SL values live
#pragma unroll
      for (int c = 0; c < SL; ++c) z[c] = sub(z[c], mulc(tw, ld<double>(vs + c)));
      lds_order();
    }
  }

  // the row from memory
  __device__ __forceinline__ void load(int row, int n, const Geom &G, int64_t base, const double *re,
                                       const double *im) {
#pragma unroll
    for (int c = 0; c < SL; ++c) {
      z[c] = mk<double>(0, 0);
      if (row < n && SL * h + c < n) {
        const int64_t idx = base + G.el(row, SL * h + c);
        z[c] = mk<double>(re[idx], im[idx]);
      }
    }
  }
  __device__ __forceinline__ void store(int row, int n, const Geom &G, int64_t base, double *re, double *im) const {
#pragma unroll
    for (int c = 0; c < SL; ++c)
      if (row < n && SL * h + c < n) {
        const int64_t idx = base + G.el(row, SL * h + c);
        re[idx] = z[c].re;
        im[idx] = z[c].im;
      }
  }

  // The ring's slots but the first (which the iteration is writing) hold
  // identities before the first phase: sweeps before the first, for the
  // segments that lag.  wave, waves: this one of the replaying wavefronts.
  __device__ __forceinline__ void start(Ring &ring, int wave, int waves) {
    __syncthreads();  // every wavefront has left its stage, which the slots share
    for (int s = 1 + wave; s < R; s += waves) ring_identity(ring, s, lane, 0);
  }

  // rotations fetched together: as many as fit beside the row
  static constexpr int kStep = SL > 24 ? 2 : 4;

  // whether any of the wavefront's rows holds an infinity or a NaN
  __device__ __forceinline__ bool any_non_finite() const {
    unsigned top = 0;
#pragma unroll
    for (int c = 0; c < SL; ++c) top = max(top, high_word(z[c]));
    return __any(top >= kNonFinite);
  }

  // replay every recorded sweep, until the one flagged last
  __device__ __forceinline__ void replay(const Ring &ring) {
    int cur = 0;
    for (;;) {
      __syncthreads();
      int sl = cur - h;  // this segment's sweep
      sl = sl < 0 ? sl + R : sl;
      const StepRec *ps = ring.step[sl] + SL * h;
      // ---- the pairs across segment borders ----
      if constexpr (NT > 1) {
        // upper border: step SL h + SL - 1 of the sweep before this
        // segment's; lower border: step SL h - 1 of this segment's sweep
        int su = sl == 0 ? R - 1 : sl - 1;
        const bool up = h + 1 < NT, dn = h > 0;
        cx<double> cu = mk<double>(1, 0), cd = mk<double>(1, 0);
        double s_u = 0.0, s_d = 0.0;
        if (up) {
          cu = ld<double>(&ring.step[su][SL * h + SL - 1].c);
          s_u = ring.step[su][SL * h + SL - 1].sr.x;
        }
        if (dn) {
          cd = ld<double>(&ps[-1].c);
          s_d = ps[-1].sr.x;
        }
        cx<double> zu = seg_shift(z[0], 1), zd = seg_shift(z[SL - 1], -1);
        const Rot<double> qu{cu, s_u}, qd{cd, s_d};
        if (up) rot_right(qu, z[SL - 1], zu);
        if (dn) rot_right(qd, zd, z[0]);
      }
      // ---- steps 0..SL-2 of each segment, kStep at a time where any is live ----
      using Mask = std::conditional_t<(SL > 32), uint64_t, unsigned>;
      Mask kmask = 0;
#pragma unroll
      for (int g = 0; g < NT; ++g) {
        const int sg = cur - g < 0 ? cur - g + R : cur - g;
        const int lo = __builtin_amdgcn_readfirstlane(ring.L[sg]) - SL * g;
        const int hi = __builtin_amdgcn_readfirstlane(ring.I[sg]) - SL * g;
        const int l = lo < 0 ? 0 : (lo > SL - 1 ? SL - 1 : lo), e = hi < 0 ? 0 : (hi > SL - 1 ? SL - 1 : hi);
        kmask |= e > l ? ((Mask(1) << e) - 1u) & ~((Mask(1) << l) - 1u) : Mask(0);
      }
      static_for<(SL + kStep - 1) / kStep>([&](auto bc) {
        constexpr int b = decltype(bc)::value * kStep;
        if ((kmask >> b) & ((1u << kStep) - 1u)) {
          constexpr int m = b + kStep < SL ? kStep : SL - 1 - b;
          if constexpr (m > 0) {
            Rot<double> q[m];
#pragma unroll
            for (int j = 0; j < m; ++j) q[j] = Rot<double>{ld<double>(&ps[b + j].c), ps[b + j].sr.x};
#pragma unroll
            for (int j = 0; j < m; ++j) rot_right(q[j], z[b + j], z[b + j + 1]);
          }
        }
      });
      // ---- H(I, I-1) made real: column I ----
#pragma unroll
      for (int g = 0; g < NT; ++g) {
        const int sg = cur - g < 0 ? cur - g + R : cur - g;
        const int ig = __builtin_amdgcn_readfirstlane(ring.I[sg]);
        if (ig > 0 && ig >= SL * g && ig < SL * g + SL) {
          const cx<double> ph = ld<double>(&ring.ph[sg]);
          const cx<double> pl = h == g ? ph : mk<double>(1, 0);
          // (a branch tree over the columns is merged back by the compiler
          // into an indexed array in scratch memory: one test per column)
#pragma unroll
          for (int k = 0; k < SL; ++k)
            if (k == ig - SL * g) z[k] = mulc(z[k], pl);
        }
      }
      const int last = __builtin_amdgcn_readfirstlane(ring.last[cur]);
      cur = cur + 1 == R ? 0 : cur + 1;
      if (last) break;
    }
  }
};

// SchurRows::replay where H or Z holds an infinity or a NaN: the steps of each
// sweep alone, not the identity at the others, which would carry such a value
// into the column beside it.  One lane to a row, in the output planes (row < 0:
// none); as many barriers as replay.
template <typename Ring>
__device__ __noinline__ void replay_rare(const Ring *ring, int row, Geom G, int64_t base, double *re, double *im) {
  for (int cur = 0;;) {
    __syncthreads();
    const int L = ring->L[cur], I = ring->I[cur];
    if (row >= 0 && I > 0) {
      auto put = [&](int c, cx<double> x) {
        re[base + G.el(row, c)] = x.re;
        im[base + G.el(row, c)] = x.im;
      };
      cx<double> z = mk<double>(re[base + G.el(row, L)], im[base + G.el(row, L)]);
      for (int K = L; K < I; ++K) {
        cx<double> next = mk<double>(re[base + G.el(row, K + 1)], im[base + G.el(row, K + 1)]);
        rot_right(Rot<double>{ld<double>(&ring->step[cur][K].c), ring->step[cur][K].sr.x}, z, next);
        put(K, z);
        z = next;
      }
      put(I, mulc(z, ld<double>(&ring->ph[cur])));
    }
    const int last = __builtin_amdgcn_readfirstlane(ring->last[cur]);
    cur = cur + 1 == Ring::R ? 0 : cur + 1;
    if (last) return;
  }
}

// --------------------------------------------------------------------------
// Eigenvectors of the triangular tile (ztrevc + backsubstitution,
// Toolbox.hpp:1133-1313, 31-136) by one wavefront, lane k solving for
// eigenvector k (and k + 64) with the reference's small-pivot clamp:
// row by row from the bottom, y(j) = (T(j,k) - sum_{i>j} T(j,i) y(i)) /
// (T(j,j) - T(k,k)), which overwrites row j of T right after its last use, so
// T and the solutions share the tile (y = -x above the diagonal).  The sums
// stay in registers: one store per entry, where the column form stores every
// partial sum.
// kRare (the tile holds an infinity or a NaN): entries that an eigenvector does
// not depend on are left out, not multiplied by a zero y.  (With the sum selected
// instead of y for every input, which lengthens its chain, ztrevc of order 64 x
// 8,192 took 1.71 ms instead of 1.65, order 96 x 1,024 1.38 instead of 1.27.)
// --------------------------------------------------------------------------
template <bool kRare, int P, typename T>
__device__ __forceinline__ void trevc_steps(const T &t, int n, int lane) {
  using R = double;
  const R ulp = limits<R>::eps;
  const R smlnum = limits<R>::tiny * (R(n > 0 ? n : 1) / ulp);
  cx<R> lam[P];
  R smin[P];
  int coff[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int k = lane + 64 * p < n ? lane + 64 * p : n - 1;
    coff[p] = t.off(k);
    lam[p] = ld<R>(t.at(k, k));
    smin[p] = fmax(ulp * cabs1(lam[p]), smlnum);
  }
  for (int j = n - 2; j >= 0; --j) {
    cx<R> acc[P];
#pragma unroll
    for (int p = 0; p < P; ++p) acc[p] = ld<R>(t.h + coff[p] + j);  // lanes k <= j: not used
#pragma unroll 4
    for (int i = j + 1; i < n - 1; ++i) {
      const cx<R> tji = ld<R>(t.at(j, i));
#pragma unroll
      for (int p = 0; p < P; ++p) {
        cx<R> y = ld<R>(t.h + coff[p] + i);
        if constexpr (kRare) {
          if (i < lane + 64 * p) acc[p] = sub(acc[p], mul(tji, y));
        } else {
          if (i >= lane + 64 * p) y = mk<R>(0, 0);
          acc[p] = sub(acc[p], mul(tji, y));
        }
      }
    }
    const cx<R> tjj = ld<R>(t.at(j, j));
    lds_order();
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int k = lane + 64 * p;
      cx<R> d = sub(tjj, lam[p]);
      if (cabs1(d) < smin[p]) d = mk(smin[p], 0.0);
      if (k > j && k < n) st<R>(t.h + coff[p] + j, mul(acc[p], inv(d)));
    }
    lds_order();
  }
}

template <int P, typename T>
__device__ __noinline__ void trevc_rare(T t, int n, int lane) {
  trevc_steps<true, P>(t, n, lane);
}

// top: the largest high word of the tile before the iteration
template <int P, typename T>
__device__ __forceinline__ void trevc_rows(const T &t, int n, int lane, unsigned top) {
  if (__builtin_expect(top >= kNonFinite, 0)) trevc_rare<P>(t, n, lane);
  else trevc_steps<false, P>(t, n, lane);
}

typedef double d4 __attribute__((ext_vector_type(4)));

// The back-transform V = Z X of ztrevc (Toolbox.hpp:1268-1275) for the RW
// rows from row0 that this wavefront holds, on the FP64 matrix cores:
// v_mfma_f64_16x16x4f64 multiplies a 16 x 4 slice of Z (A operand: lane (c, q)
// = (l % 16, l / 16) supplies Z(16 I + c, k0 + q)) by a 4 x 16 slice of X (B
// operand: X(k0 + q, 16 J + c), read from the tile, where the solve left
// y = -x above the diagonal) into a 16 x 16 block of V (lane (c, q), slot s:
// V(16 I + 4 s + q, 16 J + c)).  The complex product is four real products.
// The A operand's entry lives in another lane of its row's NT: four lane
// permutes per slice (one per q) and a select.  X is unit upper triangular:
// column block J needs the row blocks K <= J only.  The result goes straight
// to the V planes.
template <int SL, int NT, typename T>
__device__ __forceinline__ void backtransform_mfma(const T &t, const SchurRows<SL, NT> &zr, int row0, int n,
                                                   const Geom &G, int64_t base, double *rV, double *iV) {
  constexpr int RW = SchurRows<SL, NT>::RW, CAP = SchurRows<SL, NT>::CAP;
  static_assert(RW % 16 == 0, "16 x 16 blocks");
  const int lane = zr.lane, c = lane & 15, q = lane >> 4;
  // one block of V at a time (runtime loops: the row of Z takes most of the
  // registers, so only one block's accumulators stay live)
  for (int J = 0; 16 * J < n; ++J) {
    const int j = 16 * J + c;
    for (int I = 0; I < RW / 16; ++I) {
      d4 vre = d4{0, 0, 0, 0}, vim = d4{0, 0, 0, 0};
#pragma unroll
      for (int K = 0; K < (CAP + 15) / 16; ++K) {
        if (K > J) break;  // X is upper triangular
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = 16 * K + 4 * s + q;
          cx<double> x = mk<double>(k == j ? 1.0 : 0.0, 0);
          if (k < j && j < n) {
            const cx<double> y = ld<double>(t.at(k, j));
            x = mk<double>(-y.re, -y.im);
          }
          cx<double> za = mk<double>(0, 0);
#pragma unroll
          for (int qq = 0; qq < 4; ++qq) {
            const int e = 16 * K + 4 * s + qq;  // column of Z
            if (e >= CAP) continue;
            const int src = 16 * I + c + RW * (e / SL);
            const double re = __shfl(zr.z[e % SL].re, src), im = __shfl(zr.z[e % SL].im, src);
            if (qq == q) za = mk<double>(re, im);
          }
          vre = __builtin_amdgcn_mfma_f64_16x16x4f64(za.re, x.re, vre, 0, 0, 0);
          vre = __builtin_amdgcn_mfma_f64_16x16x4f64(-za.im, x.im, vre, 0, 0, 0);
          vim = __builtin_amdgcn_mfma_f64_16x16x4f64(za.re, x.im, vim, 0, 0, 0);
          vim = __builtin_amdgcn_mfma_f64_16x16x4f64(za.im, x.re, vim, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);  // one slice's operands live at a time
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int row = row0 + 16 * I + 4 * s + q;
        if (row < n && j < n) {
          const int64_t idx = base + G.el(row, j);
          rV[idx] = vre[s];
          iV[idx] = vim[s];
        }
      }
    }
  }
}

// The same for rows that hold an infinity or a NaN, which the zeros of X would
// carry into the columns before it: lane j (and j + 64) takes column j of a row
// at a time, from the V planes, which are not written yet.
template <int P, typename T>
__device__ __noinline__ void backtransform_rare(T t, int row0, int row1, int n, int lane, Geom G,
                                                int64_t base, double *rV, double *iV) {
  for (int row = row0; row < row1; ++row) {
    cx<double> acc[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int64_t idx = base + G.el(row, lane + 64 * p < n ? lane + 64 * p : 0);
      acc[p] = mk<double>(rV[idx], iV[idx]);
    }
    for (int k = 0; k + 1 < n; ++k) {
      const cx<double> z = mk<double>(rV[base + G.el(row, k)], iV[base + G.el(row, k)]);
#pragma unroll
      for (int p = 0; p < P; ++p)
        if (k < lane + 64 * p && lane + 64 * p < n) acc[p] = sub(acc[p], mul(z, ld<double>(t.at(k, lane + 64 * p))));
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
      if (lane + 64 * p < n) {
        const int64_t idx = base + G.el(row, lane + 64 * p);
        rV[idx] = acc[p].re;
        iV[idx] = acc[p].im;
      }
  }
}

}  // namespace veig
