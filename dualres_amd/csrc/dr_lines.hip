// Instances of the register line transforms (dr_lines.hpp) for the lengths of
// one part of DR_LINE_LENGTHS.  Compiled once per precision, pass and part
// (DR_LINES_T; DR_LINES_PASS 0 inverse strided, 1 forward strided, 2 leapfrog z,
// 3 rows without the residual, 4 rows with it, 5 the correlations, float64
// only, 6 whole planes; DR_LINES_PART), so that the objects build side by side
// and a process loads the device code of the lengths it uses: an object is
// loaded with its first launch, at about 1.6 ms per megabyte, and the passes
// of all lengths hold 13 of them.
#include "dr_lines.hpp"

namespace drh {

using LT = DR_LINES_T;

// m's case: the launch where m is one of this part's lengths
#define DR_CASE_IF(m, KERNEL, SHAPE, cols, ...)                                       \
  case m:                                                                             \
    if constexpr (line_part(m) == DR_LINES_PART) {                                    \
      using Sh = SHAPE;                                                               \
      const int g = cdiv(cols, Sh::COLS);                                             \
      hipLaunchKernelGGL((KERNEL), dim3(g), dim3(Sh::NT), 0, s, __VA_ARGS__);         \
      DR_HIP(hipGetLastError());                                                      \
      return g;                                                                       \
    }                                                                                 \
    return 0;
#define DR_SWITCH(M)            \
  switch (M) {                  \
    DR_LINE_LENGTHS(DR_CASE)    \
    default: return 0;          \
  }
#define DR_ARGS(...) __VA_ARGS__

#if DR_LINES_PASS == 2
template <>
int lines_z_part<DR_LINES_PART>(int M, const cx<LT>* tw, int nb, int n_in, int n_out, cx<LT>* T1,
                                const MidLeapfrog<LT>& mid, hipStream_t s) {
#define DR_CASE(m) DR_CASE_IF(m, DR_ARGS(k_zlines<LT, m>), DR_ARGS(ZShape<LT, m>), nb, tw, nb, n_in, n_out, T1, mid)
  DR_SWITCH(M)
#undef DR_CASE
}
template <>
int lines_z_kick_part<DR_LINES_PART>(int M, const cx<LT>* tw, int nb, int n_in, const cx<LT>* T1,
                                     const EpiMomentum<LT>& em, hipStream_t s) {
#define DR_CASE(m) DR_CASE_IF(m, DR_ARGS(k_zkick<LT, m>), DR_ARGS(ZShape<LT, m>), nb, tw, nb, n_in, T1, em)
  DR_SWITCH(M)
#undef DR_CASE
}
#elif DR_LINES_PASS == 5
template <>
int lines_corr_part<DR_LINES_PART>(int M, const CorrZ& a, hipStream_t s) {
#define DR_CASE(m) DR_CASE_IF(m, DR_ARGS(k_corr_z<m>), DR_ARGS(StridedShape<double, m>), a.nb, a)
  DR_SWITCH(M)
#undef DR_CASE
}
template <>
int rows_mask_part<DR_LINES_PART>(int Mh, const MaskRows& a, hipStream_t s) {
#define DR_CASE(m) DR_CASE_IF(m, DR_ARGS(k_mask_rows<m / 2>), DR_ARGS(RowShape<double, m / 2>), a.nrows, a)
  DR_SWITCH(2 * Mh)
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
// The lengths of the default embedding and three quarters of them on both
// axes, as far as plane_cap allows: a kernel for each pair, one object for all.
// Other lengths take the separate kernels; they have not been measured by
// planes.  The region's rows have to fit in the kernel's plane (they do where
// the torus is at least twice the data) and samples are fetched in pairs.
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
template <>
int lines_strided_part<DR_LINES_PART, DR_LINES_PASS == 0>(int M, const LineArgs<LT>& a, hipStream_t s) {
#define DR_CASE(m) \
  DR_CASE_IF(m, DR_ARGS(k_lines<LT, DR_LINES_PASS == 0, m>), DR_ARGS(StridedShape<LT, m>), a.ncol, a)
  DR_SWITCH(M)
#undef DR_CASE
}
#elif DR_LINES_PASS == 3
// rows: the table lists M0 = 2 Mh
template <>
int rows_c2r_part<DR_LINES_PART>(int Mh, const RowArgs<LT>& a, hipStream_t s) {
#define DR_CASE(m) DR_CASE_IF(m, DR_ARGS(k_c2r_rows<LT, m / 2>), DR_ARGS(RowShape<LT, m / 2>), a.nrows, a)
  DR_SWITCH(2 * Mh)
#undef DR_CASE
}
template <>
int rows_r2c_part<DR_LINES_PART>(int Mh, const RowArgs<LT>& a, const LoadResidual<LT>& res, hipStream_t s) {
  if (a.n0 < 2) return 0;  // samples are fetched in pairs
  const RowResidual<LT> rr{res};
#define DR_CASE(m) DR_CASE_IF(m, DR_ARGS(k_r2c_rows<LT, m / 2>), DR_ARGS(RowShape<LT, m / 2>), a.nrows, a, rr)
  DR_SWITCH(2 * Mh)
#undef DR_CASE
}
#else
template <>
int rows_residual_part<DR_LINES_PART>(int Mh, const RowArgs<LT>& a, const LoadResidual<LT>& res, hipStream_t s) {
  if (a.n0 < 2) return 0;  // samples are fetched in pairs
  const RowResidual<LT> rr{res};
#define DR_CASE(m) DR_CASE_IF(m, DR_ARGS(k_residual_rows<LT, m / 2>), DR_ARGS(RowShape<LT, m / 2>), a.nrows, a, rr)
  DR_SWITCH(2 * Mh)
#undef DR_CASE
}
#endif

}  // namespace drh
