// Instances of the register line transforms (dr_lines.hpp) for every length
// of DR_LINE_LENGTHS.  Compiled once per precision and pass (DR_LINES_T;
// DR_LINES_PASS 0 inverse strided, 1 forward strided, 2 leapfrog z, 3 rows
// without the residual, 4 rows with it, 5 the correlations, float64 only, 6
// whole planes) so the objects build side by side.
#include "dr_lines.hpp"

namespace drh {

using LT = DR_LINES_T;

#if DR_LINES_PASS == 2
int lines_z(int M, const cx<LT>* tw, int nb, int n_in, int n_out, cx<LT>* T1, const MidLeapfrog<LT>& mid,
            hipStream_t s) {
#define DR_CASE(m)                                                                                       \
  case m: {                                                                                              \
    using Sh = ZShape<LT, m>;                                                                         \
    const int g = cdiv(nb, Sh::TB);                                                                      \
    hipLaunchKernelGGL((k_zlines<LT, m>), dim3(g), dim3(Sh::NT), 0, s, tw, nb, n_in, n_out, T1, mid);    \
    DR_HIP(hipGetLastError());                                                                           \
    return g;                                                                                            \
  }
  switch (M) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
int lines_z_kick(int M, const cx<LT>* tw, int nb, int n_in, const cx<LT>* T1, const EpiMomentum<LT>& em,
                 hipStream_t s) {
#define DR_CASE(m)                                                                                       \
  case m: {                                                                                              \
    using Sh = ZShape<LT, m>;                                                                            \
    const int g = cdiv(nb, Sh::TB);                                                                      \
    hipLaunchKernelGGL((k_zkick<LT, m>), dim3(g), dim3(Sh::NT), 0, s, tw, nb, n_in, T1, em);             \
    DR_HIP(hipGetLastError());                                                                           \
    return g;                                                                                            \
  }
  switch (M) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
#elif DR_LINES_PASS == 5
int lines_corr(int M, const CorrZ& a, hipStream_t s) {
#define DR_CASE(m)                                                                                       \
  case m: {                                                                                              \
    using Sh = StridedShape<double, m>;                                                                  \
    const int g = cdiv(a.nb, Sh::TB);                                                                    \
    hipLaunchKernelGGL((k_corr_z<m>), dim3(g), dim3(Sh::NT), 0, s, a);                                   \
    DR_HIP(hipGetLastError());                                                                           \
    return g;                                                                                            \
  }
  switch (M) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
int rows_mask(int Mh, const MaskRows& a, hipStream_t s) {
#define DR_CASE(m)                                                                                       \
  case m: {                                                                                              \
    using Sh = RowShape<double, m / 2>;                                                                  \
    const int g = cdiv(a.nrows, Sh::RW);                                                                 \
    hipLaunchKernelGGL((k_mask_rows<m / 2>), dim3(g), dim3(Sh::NT), 0, s, a);                            \
    DR_HIP(hipGetLastError());                                                                           \
    return g;                                                                                            \
  }
  switch (2 * Mh) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
#elif DR_LINES_PASS == 6
template <int m0, int m1>
static bool plane_launch(int nz, const PlaneArgs<LT>& a, const RowResidual<LT>& rr, hipStream_t s) {
  if constexpr (m0 * m1 <= plane_cap<LT>()) {
    hipLaunchKernelGGL((k_plane<LT, m0 / 2, m1>), dim3(nz), dim3(kPlaneNT), 0, s, a, rr);
    DR_HIP(hipGetLastError());
    return true;
  }
  return false;
}
// the region's rows have to fit in the kernel's plane (they do where the
// torus is at least twice the data) and samples are fetched in pairs
int plane_residual(int Mh, int MY, int nz, const PlaneArgs<LT>& a, const LoadResidual<LT>& res, hipStream_t s) {
  if (a.x.n0 < 2 || a.n1 < 1 || a.n1 > MY / 2 + 1) return 0;
  const RowResidual<LT> rr{res};
#define DR_CASE(m0, m1) \
  if (2 * Mh == m0 && MY == m1) return plane_launch<m0, m1>(nz, a, rr, s) ? nz : 0;
#define DR_ROW(m0) DR_CASE(m0, 32) DR_CASE(m0, 48) DR_CASE(m0, 64) DR_CASE(m0, 96) DR_CASE(m0, 128)
  DR_ROW(32) DR_ROW(48) DR_ROW(64) DR_ROW(96) DR_ROW(128)
#undef DR_ROW
#undef DR_CASE
  return 0;
}
#elif DR_LINES_PASS < 2
#if DR_LINES_PASS == 0
int lines_inverse(int M, const LineArgs<LT>& a, hipStream_t s) {
#else
int lines_forward(int M, const LineArgs<LT>& a, hipStream_t s) {
#endif
#define DR_CASE(m)                                                                                       \
  case m: {                                                                                              \
    using Sh = StridedShape<LT, m>;                                                                         \
    const int g = cdiv(a.ncol, Sh::TB);                                                                  \
    hipLaunchKernelGGL((k_lines<LT, DR_LINES_PASS == 0, m>), dim3(g), dim3(Sh::NT), 0, s, a);            \
    DR_HIP(hipGetLastError());                                                                           \
    return g;                                                                                            \
  }
  switch (M) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
#else
// rows: the table lists M0 = 2 Mh
#define DR_ROWS(KERNEL, ...)                                                                             \
  {                                                                                                      \
    using Sh = RowShape<LT, MH>;                                                                         \
    const int g = cdiv(a.nrows, Sh::RW);                                                                 \
    hipLaunchKernelGGL((KERNEL<LT, MH>), dim3(g), dim3(Sh::NT), 0, s, __VA_ARGS__);                      \
    DR_HIP(hipGetLastError());                                                                           \
    return g;                                                                                            \
  }
#if DR_LINES_PASS == 3
int rows_c2r(int Mh, const RowArgs<LT>& a, hipStream_t s) {
#define DR_CASE(m)                     \
  case m: {                            \
    constexpr int MH = m / 2;          \
    DR_ROWS(k_c2r_rows, a)             \
  }
  switch (2 * Mh) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
int rows_r2c(int Mh, const RowArgs<LT>& a, const LoadResidual<LT>& res, hipStream_t s) {
  if (a.n0 < 2) return 0;  // samples are fetched in pairs
  const RowResidual<LT> rr{res};
#define DR_CASE(m)                     \
  case m: {                            \
    constexpr int MH = m / 2;          \
    DR_ROWS(k_r2c_rows, a, rr)         \
  }
  switch (2 * Mh) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
#else
int rows_residual(int Mh, const RowArgs<LT>& a, const LoadResidual<LT>& res, hipStream_t s) {
  if (a.n0 < 2) return 0;  // samples are fetched in pairs
  const RowResidual<LT> rr{res};
#define DR_CASE(m)                     \
  case m: {                            \
    constexpr int MH = m / 2;          \
    DR_ROWS(k_residual_rows, a, rr)    \
  }
  switch (2 * Mh) {
    DR_LINE_LENGTHS(DR_CASE)
    default: return 0;
  }
#undef DR_CASE
}
#endif
#undef DR_ROWS
#endif

}  // namespace drh
