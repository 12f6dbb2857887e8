// Line transforms held in registers, for the passes of a leapfrog step.
//
// A line of length M is transformed in two or three Stockham stages of radix
// up to 20 (LinePlan), one butterfly per thread and stage.  The first stage
// reads its elements straight from memory and the last one leaves them in the
// registers of the thread that stores them, so a transform costs one LDS
// exchange (two for three stages) with one barrier, where the tile kernels of
// dr_fft.hpp stage the tile, go through LDS twice per stage and wait twice.
// Those passes are bound by that chain of LDS round trips and barriers
// (measured per step at 168x200x180 in float32: z 81 us against 24 us of
// memory traffic), and with small tori by its latency alone.
//
// Every even 7-smooth length up to 512 has a plan (lines_length); other
// lengths, and tori past 32-bit byte offsets, keep the kernels of dr_fft.hpp.
#pragma once

#include "dr_kernels.hpp"

namespace drh {

// ---------------------------------------------------------------- butterflies
// Composite radix R = A B with A and B coprime (Good-Thomas): with
// n = (B n1 + A n2) mod R, k1 = k mod A and k2 = k mod B,
//   X[k] = sum_n1 W_A^(n1 k1) sum_n2 W_B^(n2 k2) x[n]
// has no twiddles, and both maps are compile-time permutations.
template <typename T, int A, int B, bool INV> struct DftPfa {
  static __device__ __forceinline__ void run(cx<T>* v) {
    constexpr int R = A * B;
    cx<T> t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[(B * n1 + A * n2) % R];
      Dft<T, A, INV>::run(t[n2]);
    }
    cx<T> w[A][B];
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) w[k1][n2] = t[n2][k1];
      Dft<T, B, INV>::run(w[k1]);
    }
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = w[k % A][k % B];
  }
};
template <typename T, bool INV> struct Dft<T, 6, INV> : DftPfa<T, 3, 2, INV> {};
template <typename T, bool INV> struct Dft<T, 10, INV> : DftPfa<T, 5, 2, INV> {};
template <typename T, bool INV> struct Dft<T, 12, INV> : DftPfa<T, 4, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 14, INV> : DftPfa<T, 7, 2, INV> {};
template <typename T, bool INV> struct Dft<T, 15, INV> : DftPfa<T, 5, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 20, INV> : DftPfa<T, 5, 4, INV> {};

// Radix 9 as 3 x 3 with the twiddles W9^(n2 k1), as radix 16 is 4 x 4.
struct Tw9 {  // cos and sin of 2 pi j / 9, j = 0..4
  static constexpr double c[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5,
                                  -0.93969262078590838405};
  static constexpr double s[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                                  0.34202014332566873304};
};
template <typename T, bool INV> struct Dft<T, 9, INV> {
  static __device__ __forceinline__ void run(cx<T>* v) {
    cx<T> a[3][3];  // a[n2][k1]
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
      cx<T> t[3] = {v[n2], v[n2 + 3], v[n2 + 6]};
      Dft<T, 3, INV>::run(t);
#pragma unroll
      for (int k1 = 0; k1 < 3; ++k1) {
        const int j = n2 * k1;
        a[n2][k1] = j == 0 ? t[k1] : cmul(t[k1], mk<T>((T)Tw9::c[j], INV ? (T)Tw9::s[j] : -(T)Tw9::s[j]));
      }
    }
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      cx<T> u[3] = {a[0][k1], a[1][k1], a[2][k1]};
      Dft<T, 3, INV>::run(u);
#pragma unroll
      for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = u[k2];
    }
  }
};
template <typename T, bool INV> struct Dft<T, 18, INV> : DftPfa<T, 9, 2, INV> {};

// ---------------------------------------------------------------- plans
constexpr bool line_radix(int r) {
  return r >= 2 && (r <= 10 || r == 12 || r == 14 || r == 15 || r == 16 || r == 18 || r == 20);
}
// Two stages where both radices are at most CAP, else three, the largest
// radix as small as it can be; radices in decreasing order, so that the last
// stage, whose outputs the spectral updates work on, keeps the most threads
// busy with the fewest elements each.
struct LineRadices {
  int n;
  int r[3];
};
constexpr LineRadices line_radices(int M, int cap) {
  LineRadices best{0, {1, 1, 1}};
  int bm = 1 << 20;
  for (int a = 2; a <= cap; ++a) {
    if (!line_radix(a) || M % a) continue;
    const int b = M / a;
    if (b <= a && line_radix(b) && a < bm) {
      bm = a;
      best = LineRadices{2, {a, b, 1}};
    }
  }
  if (best.n) return best;
  if (M <= cap && line_radix(M)) return LineRadices{1, {M, 1, 1}};
  for (int a = 2; a <= cap; ++a)
    for (int b = 2; b <= a; ++b) {
      if (!line_radix(a) || !line_radix(b) || M % (a * b)) continue;
      const int c = M / (a * b);
      if (c <= b && line_radix(c) && a < bm) {
        bm = a;
        best = LineRadices{3, {a, b, c}};
      }
    }
  return best;
}
template <int M, int CAP> struct LinePlan {
  static constexpr LineRadices P = line_radices(M, CAP);
  static constexpr int n = P.n;
  static_assert(n > 0, "no plan for this length");
  // radix of stage s; REV runs the stages in the opposite order, so that a
  // transform back starts on the elements the transform before it ended with
  template <bool REV> static constexpr int radix(int s) { return P.r[REV ? n - 1 - s : s]; }
  static constexpr int last = P.r[n - 1];  // of the forward order
  static constexpr int nj = M / last;      // butterflies of the widest stage (the smallest radix)
  static constexpr int rmax = P.r[0];
};

// Stage s of a line: v holds the inputs of butterfly j (elements j + r M / R)
// on entry and its outputs (elements j + r M / R after the last stage) on
// return.  at(i) is the LDS slot of element i of this thread's line; war says
// that other threads may still be reading the exchange buffer.
template <typename T, class Plan, int M, bool INV, bool REV, int TWS, int S, int NS, class At>
__device__ __forceinline__ void line_stage(cx<T>* v, int j, const cx<T>* __restrict__ tw, At&& at, bool war) {
  constexpr int R = Plan::template radix<REV>(S), BF = M / R;
  if (j < BF) Dft<T, R, INV>::run(v);
  if constexpr (S + 1 < Plan::n) {
    constexpr int R2 = Plan::template radix<REV>(S + 1), BF2 = M / R2, NS2 = NS * R;
    if (war) __syncthreads();
    if (j < BF) {
      const int jm = NS == 1 ? 0 : j % NS, d = (j - jm) * R + jm;
#pragma unroll
      for (int r = 0; r < R; ++r) *at(d + r * NS) = v[r];
    }
    __syncthreads();
    if (j < BF2) {
      const int jm = j % NS2, e = jm * (M / (NS2 * R2)) * TWS;
#pragma unroll
      for (int r = 0; r < R2; ++r) v[r] = *at(j + r * BF2);
#pragma unroll
      for (int r = 1; r < R2; ++r) {
        const cx<T> w = tw[r * e];
        v[r] = INV ? cmulc(v[r], w) : cmul(v[r], w);
      }
    }
    line_stage<T, Plan, M, INV, REV, TWS, S + 1, NS2>(v, j, tw, at, true);
  }
}
template <typename T, class Plan, int M, bool INV, bool REV, int TWS, class At>
__device__ __forceinline__ void line_fft(cx<T>* v, int j, const cx<T>* __restrict__ tw, At&& at, bool war) {
  line_stage<T, Plan, M, INV, REV, TWS, 0, 1>(v, j, tw, at, war);
}

// sum over a workgroup of NT threads, through LDS scratch of NT doubles that
// no thread reads any more; valid in thread 0
template <int NT>
__device__ __forceinline__ double line_sum(double x, double* sh) {
  const int t = threadIdx.x;
  constexpr int P2 = NT <= 64 ? 64 : NT <= 128 ? 128 : NT <= 256 ? 256 : NT <= 512 ? 512 : 1024;
  __syncthreads();
  sh[t] = x;
  __syncthreads();
  for (int s = P2 / 2; s > 0; s >>= 1) {
    if (t < s && t + s < NT) sh[t] += sh[t + s];
    __syncthreads();
  }
  return sh[0];
}

// Radix caps of the passes.  The strided passes hold one line's elements and
// nothing else, so small radices (three stages, more threads per line, 30 to
// 60 registers) hide more latency: at 1 mm the inverse y pass (320) took 19.3
// us with 8 8 5 against 23.4 with 20 16, at 1.5 mm (200) 9.9 with 8 5 5
// against 12.8 with 20 10.  The z pass also holds the state of its modes: in
// float32 it gains from fewer exchanges (84 us with 16 16 at 256x320x256, 96
// with 8 8 4), in float64 from fewer registers (240 us with 8 8 4 at
// 256x512x256, 280 with 16 16).
constexpr int kCapStrided = 10;
template <typename T> constexpr int line_cap() { return sizeof(T) == 4 ? 20 : 10; }
// columns per workgroup: runs of 128 bytes per row, more where lines are
// short, fewer where 16 lines would need over 1024 threads
template <typename T> constexpr int line_cols(int nj) { return nj < 16 || (sizeof(T) == 4 && nj <= 64) ? 16 : 8; }
template <typename T, int M, int CAP> struct LineShape {
  using Plan = LinePlan<M, CAP>;
  static constexpr int TB = line_cols<T>(Plan::nj), NT = Plan::nj * TB, COLS = TB;
  static_assert(NT <= 1024, "workgroup");
};
template <typename T, int M> using StridedShape = LineShape<T, M, kCapStrided>;
template <typename T, int M> using ZShape = LineShape<T, M, line_cap<T>()>;

// ---------------------------------------------------------------- strided lines
// Transform along an axis of ncol columns; column c = (o, b) with b < nb
// contiguous: element k of it at o * so + k * nb + b.  k_in input rows (the
// rest zero), k_out output rows.  The columns of all outer indices are tiled
// together, so that only the last tile is ragged (one column of 129 per 16
// left a ninth of the tiles nearly empty).
template <typename T> struct LineArgs {
  const cx<T>* tw;
  int nb, ncol, k_in, k_out;
  const cx<T>* src;
  long s_so;
  cx<T>* dst;
  long d_so;
  int spec;  // rows M2 of a source in the spectral state's layout (one outer index), or 0
  int wrap;  // also the last `wrap` output rows, stored after the first k_out
};
template <typename T, bool INV, int M>
__global__ void __launch_bounds__((StridedShape<T, M>::NT))
k_lines(LineArgs<T> a) {
  using Plan = typename StridedShape<T, M>::Plan;
  constexpr int TB = StridedShape<T, M>::TB, R1 = Plan::template radix<false>(0), B1 = M / R1,
                RL = Plan::template radix<false>(Plan::n - 1), BL = M / RL;
  __shared__ cx<T> buf[M * TB];
  const int b = threadIdx.x % TB, j = threadIdx.x / TB;
  const int c = xcd_tile(blockIdx.x, gridDim.x) * TB + b;
  const bool in = c < a.ncol;
  const int cc = in ? c : a.ncol - 1, o = cc / a.nb, bc = cc - o * a.nb;
  // element k of the column at s + k * sk
  const cx<T>* s = a.src + (a.spec ? Spec<T>{a.spec, a.nb}.at(0, bc) : o * a.s_so + bc);
  const int sk = a.spec ? Spec<T>::C : a.nb;
  cx<T> v[Plan::rmax];
  if (j < B1) {
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      v[r] = mk<T>(0, 0);
      if (r * B1 < a.k_in) {  // uniform; rows past the input are zero
        const int k = j + r * B1;
        const cx<T> x = s[(unsigned)(min(k, a.k_in - 1) * sk)];
        v[r].x = k < a.k_in ? x.x : (T)0;
        v[r].y = k < a.k_in ? x.y : (T)0;
      }
    }
  }
  line_fft<T, Plan, M, INV, false, 1>(v, j, a.tw, [&](int i) { return &buf[i * TB + b]; }, false);
  if (j < BL && in) {
    cx<T>* d = a.dst + (o * a.d_so + bc);
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const int k = j + r * BL;
      if (k < a.k_out) d[(unsigned)(k * a.nb)] = v[r];
      else if (k >= M - a.wrap) d[(unsigned)((k - M + a.wrap + a.k_out) * a.nb)] = v[r];
    }
  }
}

// ---------------------------------------------------------------- leapfrog z pass
// Forward transform of the n_in input rows, kick and drift of every mode,
// inverse transform, n_out rows out, in place on T1 (k_strided2_pf's work).
// The inverse runs the forward stages in the opposite order, so it starts on
// the modes the forward transform left in the thread's registers and the
// kick and drift need no exchange.  The state of the first NP modes is
// fetched before the transform, the rest in groups of 4 after it (float32, z
// pass at 168x200x180 33 us with NP = 4, 37.5 with 8, 38.5 with all 12; at
// 256x320x256 89, 88 and 86).
template <typename T> constexpr int line_np(int rl) {
  const int m = 4;
  return rl < m ? rl : m;
}
// a column's n_in input rows, the rest zero, for the first stage
template <typename T, int R1, int B1>
__device__ __forceinline__ void z_load(cx<T>* v, int j, const cx<T>* src, int nb, int n_in) {
  if (j >= B1) return;
#pragma unroll
  for (int r = 0; r < R1; ++r) {
    v[r] = mk<T>(0, 0);
    if (r * B1 < n_in) {  // uniform
      const int k = j + r * B1;
      const cx<T> x = src[(unsigned)(min(k, n_in - 1) * nb)];
      v[r].x = k < n_in ? x.x : (T)0;
      v[r].y = k < n_in ? x.y : (T)0;
    }
  }
}
template <typename T, int M>
__global__ void __launch_bounds__((ZShape<T, M>::NT))
k_zlines(const cx<T>* tw, int nb, int n_in, int n_out, cx<T>* T1, MidLeapfrog<T> mid) {
  using Plan = typename ZShape<T, M>::Plan;
  constexpr int TB = ZShape<T, M>::TB, R1 = Plan::template radix<false>(0), B1 = M / R1, RL = Plan::last,
                BL = M / RL, NT = ZShape<T, M>::NT, NP = line_np<T>(RL);
  __shared__ __align__(16) cx<T> buf[M * TB];
  static_assert(sizeof(buf) >= NT * sizeof(double), "reduction scratch");
  bind_scalars(mid);
  const int b = threadIdx.x % TB, j = threadIdx.x / TB;
  const int c = xcd_tile(blockIdx.x, gridDim.x) * TB + b;
  const bool in = c < nb;
  const int cc = in ? c : nb - 1;
  cx<T> v[Plan::rmax];
  z_load<T, R1, B1>(v, j, T1 + cc, nb, n_in);
  // mode k of the column in the state's layout
  const unsigned s0 = (unsigned)Spec<T>{M, nb}.at(0, cc);
  auto si = [&](int k) { return s0 + (unsigned)(k * Spec<T>::C); };
  typename MidLeapfrog<T>::State st[NP];
#pragma unroll
  for (int r = 0; r < NP; ++r) st[r] = mid.fetch_at(si(j + r * BL));
  auto at = [&](int i) { return &buf[i * TB + b]; };
  line_fft<T, Plan, M, false, false, 1>(v, j, tw, at, false);
  // every thread owns RL modes (BL is the widest stage); a tail column works
  // on the last one's values and stores nothing
#pragma unroll
  for (int r = 0; r < NP; ++r) v[r] = mid.apply_at(si(j + r * BL), cc, v[r], st[r], in);
#pragma unroll
  for (int r0 = NP; r0 < RL; r0 += 4) {
    typename MidLeapfrog<T>::State sr[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (r0 + u < RL) sr[u] = mid.fetch_at(si(j + (r0 + u) * BL));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (r0 + u < RL) v[r0 + u] = mid.apply_at(si(j + (r0 + u) * BL), cc, v[r0 + u], sr[u], in);
  }
  line_fft<T, Plan, M, true, true, 1>(v, j, tw, at, true);
  if (j < B1 && in) {
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int k = j + r * B1;
      if (k < n_out) T1[(unsigned)(k * nb + cc)] = v[r];
    }
  }
  if (mid.do_red) {
    const double s = line_sum<NT>(in ? mid.a0 : 0.0, reinterpret_cast<double*>(buf));
    if (threadIdx.x == 0) mid.part[blockIdx.x] = s;
  }
}

// The leapfrog's last half kick: forward transform, p's update and the end
// point's energies (EpiMomentum), nothing back.  Same shape as the z pass.
// Once per update: 64x64x32 float32 23 -> 5 us against the tile kernel, 256x512x256
// float64 251 -> 212 (281 with cached loads of the state behind a branch).
template <typename T, int M>
__global__ void __launch_bounds__((ZShape<T, M>::NT))
k_zkick(const cx<T>* tw, int nb, int n_in, const cx<T>* T1, EpiMomentum<T> em) {
  using Plan = typename ZShape<T, M>::Plan;
  constexpr int TB = ZShape<T, M>::TB, R1 = Plan::template radix<false>(0), B1 = M / R1, RL = Plan::last,
                BL = M / RL, NT = ZShape<T, M>::NT, NP = line_np<T>(RL);
  __shared__ __align__(16) cx<T> buf[M * TB];
  bind_scalars(em);
  const int b = threadIdx.x % TB, j = threadIdx.x / TB;
  const int c = xcd_tile(blockIdx.x, gridDim.x) * TB + b;
  const bool in = c < nb;
  const int cc = in ? c : nb - 1;
  cx<T> v[Plan::rmax];
  z_load<T, R1, B1>(v, j, T1 + cc, nb, n_in);
  const unsigned s0 = (unsigned)Spec<T>{M, nb}.at(0, cc);
  auto si = [&](int k) { return s0 + (unsigned)(k * Spec<T>::C); };
  typename EpiMomentum<T>::State st[NP];
#pragma unroll
  for (int r = 0; r < NP; ++r) st[r] = em.fetch_at(si(j + r * BL));
  line_fft<T, Plan, M, false, false, 1>(v, j, tw, [&](int i) { return &buf[i * TB + b]; }, false);
#pragma unroll
  for (int r0 = 0; r0 < RL; r0 += NP) {
    if (r0 > 0) {
#pragma unroll
      for (int u = 0; u < NP; ++u)
        if (r0 + u < RL) st[u] = em.fetch_at(si(j + (r0 + u) * BL));
    }
#pragma unroll
    for (int u = 0; u < NP; ++u)
      if (r0 + u < RL) em.apply_at(si(j + (r0 + u) * BL), cc, v[r0 + u], st[u], in);
  }
  double* sh = reinterpret_cast<double*>(buf);
  const double prior = line_sum<NT>(em.a0, sh);
  if (threadIdx.x == 0) em.part_prior[blockIdx.x] = prior;
  const double kin = line_sum<NT>(em.a1, sh);
  if (threadIdx.x == 0) em.part_kin[blockIdx.x] = kin;
}

// ---------------------------------------------------------------- rows along x
// Real rows of length M0 = 2 Mh as complex lines of length Mh on packed
// samples z[n] = (x[2n], x[2n+1]).  Lanes run along the row; workgroups of
// about one wavefront, so the exchange's barriers cost nothing and a few
// thousand rows spread over all CUs.  Each element of a half spectrum is
// read twice (X[k] and X[Mh - k] meet in Z[k] and Z[Mh - k]), the second time
// from the cache, in place of an exchange.
template <typename T, int Mh> struct RowShape {
  using Plan = LinePlan<Mh, line_cap<T>()>;
  static constexpr int RW = Plan::nj >= 64 ? 1 : 64 / Plan::nj, NT = RW * Plan::nj, COLS = RW;
  static constexpr int R1 = Plan::P.r[0];
  // a pad slot after every R1 elements where R1 is even: the first stage
  // writes at stride R1, which then hits every bank
  static constexpr int pad(int i) { return R1 % 2 == 0 ? i + i / R1 : i; }
  static constexpr int P = pad(Mh) + 1;  // Mh + 1 elements
};

// two neighbouring samples of a row, at any alignment of T
template <typename T> struct Pair { T a, b; };
template <typename V, typename T>
__device__ __forceinline__ Pair<T> ld_pair(const T* p) {
  typedef V U __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  const U x = *reinterpret_cast<const U*>(p);
  return Pair<T>{x[0], x[1]};
}

// half spectrum row -> Z[k] for the inverse transform (k_c2r_x's merge)
template <typename T, int Mh>
__device__ __forceinline__ cx<T> row_merge(const cx<T>* __restrict__ X, const cx<T>* __restrict__ tw, int k) {
  const cx<T> a = X[k], c = X[Mh - k];
  const cx<T> s = a + conj(c), t = cmulc(a - conj(c), tw[k]);
  return mk<T>(s.x - t.y, s.y + t.x);
}

// Z[k] and Z[Mh - k] -> X[k] of the half spectrum (k_r2c_x's split)
template <typename T>
__device__ __forceinline__ cx<T> row_split(cx<T> zk, cx<T> zm, cx<T> w) {
  const cx<T> zc = conj(zm), e = (zk + zc) * (T)0.5, d = zk - zc;
  return e + cmul(w, mk<T>(d.y * (T)0.5, -d.x * (T)0.5));
}

// residual of samples 2n, 2n + 1 (LoadResidual's arithmetic) from their mu
template <typename T>
struct RowResidual {
  LoadResidual<T> q;
  // inputs of a pair: the samples x0, x0 + 1 with x0 = 2n, or n0 - 2 where the
  // row ends (odd n0), whose second sample is then the pair's first
  struct In { Pair<T> y, r, w, wb; uint8_t m0, m1; };
  template <bool MU>
  __device__ __forceinline__ In fetch(int row, int n) const {
    In v;
    const long g = (long)row * q.n0 + min(2 * n, q.n0 - 2);
    v.m0 = q.mask[g];
    v.m1 = q.mask[g + 1];
    v.y = ld_pair<T>(q.Yg + g);
    v.r = v.w = v.wb = Pair<T>{0, 0};
    if (MU) v.r = ld_pair<T>(q.R + g);
    if (q.WTv) v.w = ld_pair<T>(q.WTv + g);
    if (q.WTvb) v.wb = ld_pair<T>(q.WTvb + g);
    return v;
  }
  __device__ __forceinline__ T one(bool m, T y, T mu, T w, T wb) {
    if (!m) return (T)0;
    const T d = y - mu;
    q.acc += (double)d * (double)d;
    T r = q.sig * d;
    if (q.WTv) r += w;
    if (q.WTvb) r += wb;
    return r;
  }
  // mu: the pair's samples (from the line) or null (from In::r)
  __device__ __forceinline__ cx<T> apply(const In& v, int n, bool row_ok, const cx<T>* mu) {
    const int x = 2 * n;
    const bool a = row_ok && x < q.n0, b = row_ok && x + 1 < q.n0, tail = x == q.n0 - 1;
    const T ya = tail ? v.y.b : v.y.a, ra = mu ? mu->x : tail ? v.r.b : v.r.a, rb = mu ? mu->y : v.r.b;
    return mk<T>(one(a && (tail ? v.m1 : v.m0), ya, ra, tail ? v.w.b : v.w.a, tail ? v.wb.b : v.wb.a),
                 one(b && v.m1, v.y.b, rb, v.w.b, v.wb.b));
  }
};

// forward transform's tail: the outputs Z[j + r BF] in v meet their mirror
// images through LDS; X[0..Mh] of the row to dst
template <typename T, int Mh, int R, class At>
__device__ __forceinline__ void row_store_split(const cx<T>* v, int j, const cx<T>* __restrict__ tw, At&& at, bool ok,
                                                cx<T>* dst) {
  constexpr int BF = Mh / R;
  __syncthreads();  // the last stage's reads of the exchange buffer
  if (j < BF) {
#pragma unroll
    for (int r = 0; r < R; ++r) *at(j + r * BF) = v[r];
  }
  __syncthreads();
  if (j < BF && ok) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int k = j + r * BF;
      dst[k] = row_split(v[r], *at(k == 0 ? 0 : Mh - k), tw[k]);
    }
    if (j == 0) dst[Mh] = row_split(v[0], v[0], tw[Mh]);
  }
}

template <typename T> struct RowArgs {
  const cx<T>* tw;  // length-M0 table
  int nrows, n0;    // rows; samples kept per row
  const cx<T>* src; // half spectra in (row pitch Mh + 1)
  cx<T>* dst;       // half spectra out
  T* R;             // mu out, or null
  T scale;          // 1 / N
};

// One row of a group whose lanes run along it: j counts the row's threads
// (plan nj of them), at(i) is the LDS slot of element i, X the half spectrum
// read and D the one written (which may be X), row the row's number in the
// region; ok is false for a lane past the last row, which works on a row it
// must not store to.
// half spectrum -> scaled samples
template <typename T, int Mh, class At>
__device__ __forceinline__ void row_inverse(const RowArgs<T>& a, const cx<T>* X, int row, int j, bool ok, At&& at,
                                            bool war) {
  using Plan = typename RowShape<T, Mh>::Plan;
  constexpr int R1 = Plan::template radix<false>(0), B1 = Mh / R1, RL = Plan::last, BL = Mh / RL;
  cx<T> v[Plan::rmax];
  if (j < B1) {
#pragma unroll
    for (int r = 0; r < R1; ++r) v[r] = row_merge<T, Mh>(X, a.tw, j + r * B1);
  }
  line_fft<T, Plan, Mh, true, false, 2>(v, j, a.tw, at, war);
  if (j < BL && ok) {
    T* d = a.R + (long)row * a.n0;
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const int x = 2 * (j + r * BL);
      if (x < a.n0) d[x] = v[r].x * a.scale;
      if (x + 1 < a.n0) d[x + 1] = v[r].y * a.scale;
    }
  }
}

// residual of the row's samples -> half spectrum
template <typename T, int Mh, class At>
__device__ __forceinline__ void row_forward(const RowArgs<T>& a, RowResidual<T>& res, cx<T>* D, int row, int j,
                                            bool ok, At&& at, bool war) {
  using Plan = typename RowShape<T, Mh>::Plan;
  constexpr int R1 = Plan::template radix<false>(0), B1 = Mh / R1, RL = Plan::last;
  cx<T> v[Plan::rmax];
  if (j < B1) {
#pragma unroll
    for (int r0 = 0; r0 < R1; r0 += 4) {
      typename RowResidual<T>::In in[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (r0 + u < R1 && 2 * (r0 + u) * B1 < a.n0) in[u] = res.template fetch<true>(row, j + (r0 + u) * B1);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (r0 + u < R1) {
          v[r0 + u] = mk<T>(0, 0);
          if (2 * (r0 + u) * B1 < a.n0) v[r0 + u] = res.apply(in[u], j + (r0 + u) * B1, ok, nullptr);
        }
    }
  }
  line_fft<T, Plan, Mh, false, false, 2>(v, j, a.tw, at, war);
  row_store_split<T, Mh, RL>(v, j, a.tw, at, ok, D);
}

// half spectrum -> samples -> residual -> half spectrum: without W the
// likelihood is local to a row.  mu goes to R only where it is asked for.
// The way back runs the stages in the opposite order, so it starts on the
// samples the inverse transform left in the thread's registers.
template <typename T, int Mh, class At>
__device__ __forceinline__ void row_residual(const RowArgs<T>& a, RowResidual<T>& res, const cx<T>* X, cx<T>* D,
                                             int row, int j, bool ok, At&& at, bool war) {
  using Plan = typename RowShape<T, Mh>::Plan;
  constexpr int R1 = Plan::template radix<false>(0), B1 = Mh / R1, RL = Plan::last, BL = Mh / RL;
  cx<T> v[Plan::rmax];
  if (j < B1) {
#pragma unroll
    for (int r = 0; r < R1; ++r) v[r] = row_merge<T, Mh>(X, a.tw, j + r * B1);
  }
  line_fft<T, Plan, Mh, true, false, 2>(v, j, a.tw, at, war);
  // BL is the widest stage: every thread owns RL packed samples
#pragma unroll
  for (int r0 = 0; r0 < RL; r0 += 4) {
    typename RowResidual<T>::In in[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (r0 + u < RL && 2 * (r0 + u) * BL < a.n0) in[u] = res.template fetch<false>(row, j + (r0 + u) * BL);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (r0 + u < RL) {
        const int n = j + (r0 + u) * BL;
        cx<T> m = v[r0 + u];
        m = m * a.scale;
        v[r0 + u] = mk<T>(0, 0);
        if (2 * (r0 + u) * BL < a.n0) {
          if (a.R && ok) {
            T* d = a.R + (long)row * a.n0;
            if (2 * n < a.n0) d[2 * n] = m.x;
            if (2 * n + 1 < a.n0) d[2 * n + 1] = m.y;
          }
          v[r0 + u] = res.apply(in[u], n, ok, &m);
        }
      }
  }
  line_fft<T, Plan, Mh, false, true, 2>(v, j, a.tw, at, true);
  row_store_split<T, Mh, R1>(v, j, a.tw, at, ok, D);
}

template <typename T, int Mh>
__global__ void __launch_bounds__((RowShape<T, Mh>::NT)) k_c2r_rows(RowArgs<T> a) {
  using Sh = RowShape<T, Mh>;
  __shared__ cx<T> buf[Sh::RW * Sh::P];
  const int j = threadIdx.x % Sh::Plan::nj, l = threadIdx.x / Sh::Plan::nj;
  const int row = blockIdx.x * Sh::RW + l, rc = min(row, a.nrows - 1);
  row_inverse<T, Mh>(a, a.src + (long)rc * (Mh + 1), rc, j, row < a.nrows,
                     [&](int i) { return &buf[l * Sh::P + Sh::pad(i)]; }, false);
}

template <typename T, int Mh>
__global__ void __launch_bounds__((RowShape<T, Mh>::NT)) k_r2c_rows(RowArgs<T> a, RowResidual<T> res) {
  using Sh = RowShape<T, Mh>;
  __shared__ __align__(16) cx<T> buf[Sh::RW * Sh::P < Sh::NT ? Sh::NT : Sh::RW * Sh::P];
  bind_scalars(res.q);
  const int j = threadIdx.x % Sh::Plan::nj, l = threadIdx.x / Sh::Plan::nj;
  const int row = blockIdx.x * Sh::RW + l, rc = min(row, a.nrows - 1);
  row_forward<T, Mh>(a, res, a.dst + (long)rc * (Mh + 1), rc, j, row < a.nrows,
                     [&](int i) { return &buf[l * Sh::P + Sh::pad(i)]; }, false);
  if (res.q.part) {
    const double s = line_sum<Sh::NT>(res.q.acc, reinterpret_cast<double*>(buf));
    if (threadIdx.x == 0) res.q.part[blockIdx.x] = s;
  }
}

template <typename T, int Mh>
__global__ void __launch_bounds__((RowShape<T, Mh>::NT)) k_residual_rows(RowArgs<T> a, RowResidual<T> res) {
  using Sh = RowShape<T, Mh>;
  __shared__ __align__(16) cx<T> buf[Sh::RW * Sh::P < Sh::NT ? Sh::NT : Sh::RW * Sh::P];
  bind_scalars(res.q);
  const int j = threadIdx.x % Sh::Plan::nj, l = threadIdx.x / Sh::Plan::nj;
  const int row = blockIdx.x * Sh::RW + l, rc = min(row, a.nrows - 1);
  row_residual<T, Mh>(a, res, a.src + (long)rc * (Mh + 1), a.dst + (long)rc * (Mh + 1), rc, j, row < a.nrows,
                      [&](int i) { return &buf[l * Sh::P + Sh::pad(i)]; }, false);
  if (res.q.part) {
    const double s = line_sum<Sh::NT>(res.q.acc, reinterpret_cast<double*>(buf));
    if (threadIdx.x == 0) res.q.part[blockIdx.x] = s;
  }
}

// ---------------------------------------------------------------- planes
// The inverse y and x passes, the single-resolution residual and the forward
// x and y passes of one z plane in one workgroup, the plane's region rows in
// LDS.  The three kernels it stands for take 4 to 5 us each at these sizes,
// launch and memory latency and little else; one kernel waits once.  A plane
// is one compute unit's work, so it only pays while that is little: us per
// update of 25 steps, separate passes and planes, float32: 32x32x32 568 and
// 381, 64x64x64 626 and 493, 64x128x64 692 and 520, 128x64x64 684 and 570,
// 128x128x64 732 and 752; float64: 540 and 400, 641 and 586, 701 and 680, 706
// and 765, 861 and 1175.  Hence the caps on M0 M1.  (The inverse and the
// forward half by planes around the products with W: no gain.)
template <typename T> constexpr int plane_cap() { return sizeof(T) == 4 ? 8192 : 4096; }
constexpr int kPlaneNT = 576;  // 9 wavefronts: 36 lines of 16 threads, 72 of 8
template <typename T> struct PlaneArgs {
  const cx<T>* twy;  // length-MY table
  int n1;            // region rows per plane
  cx<T>* T1;         // planes of MY rows of Mh + 1, in and out
  RowArgs<T> x;
};
template <typename T, int Mh, int MY> struct PlaneShape {
  using Plan = LinePlan<MY, 16>;
  using Row = RowShape<T, Mh>;
  static constexpr int LY = kPlaneNT / Plan::nj, LX = kPlaneNT / Row::Plan::nj;
  static_assert(kPlaneNT % Plan::nj == 0 && kPlaneNT % Row::Plan::nj == 0, "whole lines");
  static constexpr int EY = MY * LY, EX = LX * Row::P;
  static constexpr int E = EY > EX ? EY : EX;    // exchange buffer
  static constexpr int rows = MY / 2 + 1;        // region rows a torus of twice the data holds
  static_assert(E * sizeof(cx<T>) >= kPlaneNT * sizeof(double), "reduction scratch");
  static_assert((E + rows * (Mh + 1)) * sizeof(cx<T>) <= 160 * 1024, "LDS");
};
template <typename T, int Mh, int MY>
__global__ void __launch_bounds__(kPlaneNT) k_plane(PlaneArgs<T> a, RowResidual<T> res) {
  using Sh = PlaneShape<T, Mh, MY>;
  using Plan = typename Sh::Plan;
  using Row = typename Sh::Row;
  constexpr int H0 = Mh + 1, R1 = Plan::template radix<false>(0), B1 = MY / R1, RL = Plan::last, BL = MY / RL;
  __shared__ __align__(16) cx<T> buf[Sh::E];
  __shared__ __align__(16) cx<T> plane[Sh::rows * H0];
  bind_scalars(res.q);
  const int z = blockIdx.x, t = threadIdx.x;
  cx<T>* P = a.T1 + (long)z * MY * H0;
  const int b = t % Sh::LY, jy = t / Sh::LY;
  auto aty = [&](int i) { return &buf[i * Sh::LY + b]; };
  for (int c0 = 0; c0 < H0; c0 += Sh::LY) {
    const int c = c0 + b, cc = min(c, H0 - 1);
    cx<T> v[Plan::rmax];
    if (jy < B1) {
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = P[(jy + r * B1) * H0 + cc];
    }
    line_fft<T, Plan, MY, true, false, 1>(v, jy, a.twy, aty, c0 > 0);
    if (jy < BL && c < H0) {
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        const int k = jy + r * BL;
        if (k < a.n1) plane[k * H0 + c] = v[r];
      }
    }
  }
  __syncthreads();
  const int jx = t % Row::Plan::nj, l = t / Row::Plan::nj;
  auto atx = [&](int i) { return &buf[l * Row::P + Row::pad(i)]; };
  for (int r0 = 0; r0 < a.n1; r0 += Sh::LX) {
    const int y = r0 + l, yc = min(y, a.n1 - 1), row = z * a.n1 + yc;
    cx<T>* X = plane + yc * H0;
    row_residual<T, Mh>(a.x, res, X, X, row, jx, y < a.n1, atx, true);
  }
  __syncthreads();
  for (int c0 = 0; c0 < H0; c0 += Sh::LY) {
    const int c = c0 + b, cc = min(c, H0 - 1);
    cx<T> v[Plan::rmax];
    if (jy < B1) {
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        const int k = jy + r * B1;
        v[r] = mk<T>(0, 0);
        if (r * B1 < a.n1) {  // uniform; rows past the region are zero
          const cx<T> x = plane[min(k, a.n1 - 1) * H0 + cc];
          v[r].x = k < a.n1 ? x.x : (T)0;
          v[r].y = k < a.n1 ? x.y : (T)0;
        }
      }
    }
    line_fft<T, Plan, MY, false, false, 1>(v, jy, a.twy, aty, true);
    if (jy < BL && c < H0) {
#pragma unroll
      for (int r = 0; r < RL; ++r) P[(jy + r * BL) * H0 + c] = v[r];
    }
  }
  if (res.q.part) {
    const double s = line_sum<kPlaneNT>(res.q.acc, reinterpret_cast<double*>(buf));
    if (t == 0) res.q.part[z] = s;
  }
}

// ---------------------------------------------------------------- correlations
// Cross-correlations of an image x and its presence indicator m on a padded
// torus (dr_mce.hip).  Rows: real samples of x (0 where missing) and m to half
// spectra.
struct MaskRows {
  const cx<double>* tw;  // length-M0 table
  int nrows, nx;
  const double* img;     // rows of nx samples; 0 and NaN are missing
  cx<double>*x, *m;      // half spectra out, row pitch Mh + 1
};
template <int Mh>
__global__ void __launch_bounds__((RowShape<double, Mh>::NT)) k_mask_rows(MaskRows a) {
  using Sh = RowShape<double, Mh>;
  using Plan = typename Sh::Plan;
  constexpr int R1 = Plan::template radix<false>(0), B1 = Mh / R1, RL = Plan::last;
  __shared__ cx<double> buf[Sh::RW * Sh::P];
  const int j = threadIdx.x % Plan::nj, l = threadIdx.x / Plan::nj;
  const int row = blockIdx.x * Sh::RW + l;
  const bool ok = row < a.nrows;
  const double* q = a.img + (long)(ok ? row : a.nrows - 1) * a.nx;
  cx<double> raw[R1], v[Plan::rmax];
  if (j < B1) {
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int x = 2 * (j + r * B1);
      raw[r] = mk<double>(x < a.nx ? q[x] : 0.0, x + 1 < a.nx ? q[x + 1] : 0.0);
      if (raw[r].x != raw[r].x) raw[r].x = 0.0;
      if (raw[r].y != raw[r].y) raw[r].y = 0.0;
      v[r].x = raw[r].x;
      v[r].y = raw[r].y;
    }
  }
  auto at = [&](int i) { return &buf[l * Sh::P + Sh::pad(i)]; };
  line_fft<double, Plan, Mh, false, false, 2>(v, j, a.tw, at, false);
  row_store_split<double, Mh, RL>(v, j, a.tw, at, ok, a.x + (long)row * (Mh + 1));
  if (j < B1) {
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      v[r].x = raw[r].x != 0.0 ? 1.0 : 0.0;
      v[r].y = raw[r].y != 0.0 ? 1.0 : 0.0;
    }
  }
  line_fft<double, Plan, Mh, false, false, 2>(v, j, a.tw, at, true);
  row_store_split<double, Mh, RL>(v, j, a.tw, at, ok, a.m + (long)row * (Mh + 1));
}

// z lines: both fields forward, the products conj(X) X, conj(X) M, conj(M) M of
// every mode, each back to the rows k < k_out and the last `wrap` ones.  One
// pass over the two fields in place of two forward passes, a product pass and
// four full inverse ones (x-m and m-x are one field read at p and -p).
struct CorrZ {
  const cx<double>* tw;
  int nb, k_in, k_out, wrap;
  const cx<double>*x, *m;  // k_in rows of nb columns
  cx<double>* out[3];      // k_out + wrap rows
};
template <int M>
__global__ void __launch_bounds__((StridedShape<double, M>::NT)) k_corr_z(CorrZ a) {
  using T = double;
  using Plan = typename StridedShape<T, M>::Plan;
  constexpr int TB = StridedShape<T, M>::TB, R1 = Plan::template radix<false>(0), B1 = M / R1, RL = Plan::last;
  __shared__ cx<T> buf[M * TB];
  const int b = threadIdx.x % TB, j = threadIdx.x / TB;
  const int c = xcd_tile(blockIdx.x, gridDim.x) * TB + b;
  const bool in = c < a.nb;
  const int cc = in ? c : a.nb - 1;
  auto at = [&](int i) { return &buf[i * TB + b]; };
  cx<T> f[2][RL];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const cx<T>* s = (q ? a.m : a.x) + cc;
    cx<T> v[Plan::rmax];
    if (j < B1) {
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        v[r] = mk<T>(0, 0);
        if (r * B1 < a.k_in) {
          const int k = j + r * B1;
          const cx<T> x = s[(unsigned)(min(k, a.k_in - 1) * a.nb)];
          v[r].x = k < a.k_in ? x.x : (T)0;
          v[r].y = k < a.k_in ? x.y : (T)0;
        }
      }
    }
    line_fft<T, Plan, M, false, false, 1>(v, j, a.tw, at, q > 0);
#pragma unroll
    for (int r = 0; r < RL; ++r) f[q][r] = v[r];
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    cx<T> v[Plan::rmax];
#pragma unroll
    for (int r = 0; r < RL; ++r) v[r] = cmulc(f[p > 0][r], f[p > 1][r]);
    line_fft<T, Plan, M, true, true, 1>(v, j, a.tw, at, true);
    if (j < B1 && in) {
      cx<T>* d = a.out[p] + cc;
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        const int k = j + r * B1;
        if (k < a.k_out) d[(unsigned)(k * a.nb)] = v[r];
        else if (k >= M - a.wrap) d[(unsigned)((k - M + a.wrap + a.k_out) * a.nb)] = v[r];
      }
    }
  }
}

// ---------------------------------------------------------------- host side
// The lengths with kernels and the part of them an object of dr_lines.hip holds.
#define DR_LINE_LENGTHS(X)                                                                                           \
  X(8) X(10) X(12) X(14) X(16) X(18) X(20) X(24) X(28) X(30) X(32) X(36) X(40) X(42) X(48) X(50) X(54) X(56) X(60)    \
  X(64) X(70) X(72) X(80) X(84) X(90) X(96) X(98) X(100) X(108) X(112) X(120) X(126) X(128) X(140) X(144) X(150)      \
  X(160) X(162) X(168) X(180) X(192) X(196) X(200) X(210) X(216) X(224) X(240) X(250) X(252) X(256) X(270) X(280)     \
  X(288) X(294) X(300) X(320) X(324) X(336) X(350) X(360) X(378) X(384) X(392) X(400) X(420) X(432) X(448) X(450)     \
  X(480) X(486) X(490) X(500) X(504) X(512)
constexpr int kLineParts = 6;
constexpr int line_part(int M) { return M <= 48 ? 0 : M <= 96 ? 1 : M <= 150 ? 2 : M <= 240 ? 3 : M <= 336 ? 4 : 5; }
template <class F>
inline int with_line_part(int M, F&& f) {
  switch (line_part(M)) {
    case 0: return f(std::integral_constant<int, 0>{});
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    default: return f(std::integral_constant<int, 5>{});
  }
}
#define DR_PART(M, call) with_line_part(M, [&](auto p) { constexpr int P = decltype(p)::value; return call; })

// Each returns the number of workgroups launched, 0 when no kernel was built
// for the length (the caller then takes the kernels of dr_fft.hpp).
#define DR_LINE_API(T)                                                                                               \
  template <int P, bool INV> int lines_strided_part(int M, const LineArgs<T>& a, hipStream_t s);                     \
  template <int P> int lines_z_part(int M, const cx<T>* tw, int nb, int n_in, int n_out, cx<T>* T1,                  \
                                    const MidLeapfrog<T>& mid, hipStream_t s);                                       \
  template <int P> int lines_z_kick_part(int M, const cx<T>* tw, int nb, int n_in, const cx<T>* T1,                  \
                                         const EpiMomentum<T>& em, hipStream_t s);                                   \
  template <int P> int rows_c2r_part(int Mh, const RowArgs<T>& a, hipStream_t s);                                    \
  template <int P> int rows_r2c_part(int Mh, const RowArgs<T>& a, const LoadResidual<T>& res, hipStream_t s);        \
  template <int P> int rows_residual_part(int Mh, const RowArgs<T>& a, const LoadResidual<T>& res, hipStream_t s);   \
  inline int lines_inverse(int M, const LineArgs<T>& a, hipStream_t s) {                                             \
    return DR_PART(M, (lines_strided_part<P, true>(M, a, s)));                                                       \
  }                                                                                                                  \
  inline int lines_forward(int M, const LineArgs<T>& a, hipStream_t s) {                                             \
    return DR_PART(M, (lines_strided_part<P, false>(M, a, s)));                                                      \
  }                                                                                                                  \
  inline int lines_z(int M, const cx<T>* tw, int nb, int n_in, int n_out, cx<T>* T1, const MidLeapfrog<T>& mid,      \
                     hipStream_t s) {                                                                                \
    return DR_PART(M, lines_z_part<P>(M, tw, nb, n_in, n_out, T1, mid, s));                                          \
  }                                                                                                                  \
  inline int lines_z_kick(int M, const cx<T>* tw, int nb, int n_in, const cx<T>* T1, const EpiMomentum<T>& em,       \
                          hipStream_t s) {                                                                           \
    return DR_PART(M, lines_z_kick_part<P>(M, tw, nb, n_in, T1, em, s));                                             \
  }                                                                                                                  \
  inline int rows_c2r(int Mh, const RowArgs<T>& a, hipStream_t s) {                                                  \
    return DR_PART(2 * Mh, rows_c2r_part<P>(Mh, a, s));                                                              \
  }                                                                                                                  \
  inline int rows_r2c(int Mh, const RowArgs<T>& a, const LoadResidual<T>& res, hipStream_t s) {                      \
    return DR_PART(2 * Mh, rows_r2c_part<P>(Mh, a, res, s));                                                         \
  }                                                                                                                  \
  inline int rows_residual(int Mh, const RowArgs<T>& a, const LoadResidual<T>& res, hipStream_t s) {                 \
    return DR_PART(2 * Mh, rows_residual_part<P>(Mh, a, res, s));                                                    \
  }                                                                                                                  \
  int plane_residual(int Mh, int MY, int nz, const PlaneArgs<T>& a, const LoadResidual<T>& res, hipStream_t s);
DR_LINE_API(float)
DR_LINE_API(double)
#undef DR_LINE_API
template <int P> int rows_mask_part(int Mh, const MaskRows& a, hipStream_t s);
template <int P> int lines_corr_part(int M, const CorrZ& a, hipStream_t s);
inline int rows_mask(int Mh, const MaskRows& a, hipStream_t s) {
  return DR_PART(2 * Mh, rows_mask_part<P>(Mh, a, s));
}
inline int lines_corr(int M, const CorrZ& a, hipStream_t s) { return DR_PART(M, lines_corr_part<P>(M, a, s)); }
#undef DR_PART

}  // namespace drh
