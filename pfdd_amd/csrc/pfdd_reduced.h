// pfdd_reduced.h -- arguments and launchers of the reduced-basis kernels
// (pfdd_reduced.hpp holds the kernels and says what they compute;
// pfdd_reduced.hip is compiled once per component count R and kind so that the
// instantiations build in parallel).
#pragma once
#include "pfdd_kernels.hpp"

namespace pfdd {

constexpr int RED_MAXR = 6;
constexpr int RED_RL = 16;  // radix limit of these kernels' transforms

// What the row kernel needs of the step (by value, read through the scalar cache).
struct RedArgs {
  long P;
  int S;
  int nblk;                    // row blocks per field
  double uq2, two_pi, inv_n;
  double cd2[MAXS], asf_pi[MAXS], dslip[MAXS];
  double al[MAXS][RED_MAXR];   // e_a = sum_t al[a][t] h_t
  const double2* tau;          // per field: (tau, rate)
};
// Options of the general variant (OPT): frozen points, per-point shear, the
// prologue's extra force (virtualevolv G.c:1426-1447, per field in real
// space), and the projection alone (the prologue: no inverse transform, no
// update).  Null pointers switch the first three off.
template <typename T> struct RedOpt {
  const uint8_t* mask;
  const double* taupp;
  const cx<T>* extra;
  int project;
};

// Shapes of the row kernels (see there).
constexpr int red_unrolled(int R) { return R <= 3 ? 4 : R == 4 ? 8 : 0; }  // most fields of k_row_red
constexpr int red_ppt(bool fp64, int n, int R) { return n <= 64 || R > 3 ? 1 : fp64 || R == 3 ? 2 : 4; }
constexpr int red_rows(int n, int ppt) {
  if (n < 32) return 128 / n;
  const int pts = n % 3 == 0 ? 192 * ppt : ppt == 4 ? 512 : 256;  // points per block
  return n <= 64 ? 4 : pts / n > 0 ? pts / n : 1;
}
// rows per block for ns fields in R components
constexpr int red_row_rows(bool fp64, int n, int R, int ns) {
  return red_rows(n, ns <= red_unrolled(R) ? red_ppt(fp64, n, R) : 1);
}

// The per-field sums that ride along with the N2 pass and the column kernel.
constexpr int FOLD_ABOVE = 512;
struct FoldJob {
  const double* in;  // [F][nblk], null: nothing to fold
  double* out;       // [F][FOLD]
  int nblk, F;
};
struct FinishJob {
  const double* in;  // [F][nblk], null: the sums are finished elsewhere
  double* out;       // history
  int* step_ctr;
  int nblk, F, S;
};


template <typename T> struct RedRowLaunch {
  RedArgs a;
  RedOpt<T> o;
  cx<T>* W;
  const cx<T>* tw;
  double* partials;
  const int* step_ctr;
  unsigned nblk, batch;
  hipStream_t stream;
};
template <typename T> struct RedColLaunch {
  cx<T>* W;
  const ElasticConsts* ec;
  const T* Kst;  // stored K(k), or null: recomputed
  long P;
  const cx<T>* tw;
  unsigned batch;
  FinishJob fin;
  hipStream_t stream;
};
template <typename T> struct RedPass2Launch {
  cx<T>* W;
  long outer, inner;
  int sign;
  const cx<T>* tw;
  FoldJob fold;
  hipStream_t stream;
};
// The plane kernel (k_plane_red): its limits, its launch for planes within
// them, and where it is the faster form: a block walks its plane alone, so that
// large planes lose when there are few of them (us a step, three kernels
// against it; components x planes: 2048 x 32 17.9 and 17.6, 3072 x 32 18.5 and
// 21.2, 5120 x 64 25.4 and 26.7, but 2048 x 128 27.2 and 23.1, 4096 x 128 28.7
// and 23.4, 3072 x 512 68 and 50).
constexpr int PLANE_MAX_POINTS = 1024;
inline bool plane_faster(int n1, int n2, int R, long planes) { return n1 * n2 * R <= 2048 || planes >= 128; }
constexpr int plane_max_threads(bool fp64) { return fp64 ? 512 : 768; }
constexpr int plane_rl(bool fp64, int n1) { return fp64 && n1 >= 128 ? 8 : RED_RL; }
int plane_threads(bool fp64, int n1, int n2, int R);
size_t plane_lds(bool fp64, int n1, int n2, int R);
bool plane_fits(bool fp64, int n1, int n2, int R);
template <typename T> struct RedPlaneLaunch {
  cx<T>* W;
  const ElasticConsts* ec;
  const T* Kst;
  int n3, R;
  const cx<T>*tw1, *tw2;
  unsigned batch;
  FinishJob fin;
  hipStream_t stream;
};
bool red_plane_d(const RedPlaneLaunch<double>&, int n1, int n2);
bool red_plane_f(const RedPlaneLaunch<float>&, int n1, int n2);
bool red_pass2_d(const RedPass2Launch<double>&, int n2);
bool red_pass2_f(const RedPass2Launch<float>&, int n2);
bool red_pass2_attr(int n2);  // LDS limits of both, once per context
// One function per R; each returns false where the length is not instantiated.
#define PFDD_RED_DECL(R)                                           \
  bool red_row_d##R(const RedRowLaunch<double>&, Master<double>, int n3); \
  bool red_row_c##R(const RedRowLaunch<float>&, MasterF32C, int n3);      \
  bool red_row_l##R(const RedRowLaunch<float>&, MasterF32L, int n3);      \
  bool red_col_d##R(const RedColLaunch<double>&, int n1);                 \
  bool red_col_f##R(const RedColLaunch<float>&, int n1);                  \
  bool red_col_attr##R(int n1);  /* LDS limits of both, once per context */ \
  void red_build_d##R(double* Kst, const ElasticConsts* ec, long P, hipStream_t);  \
  void red_build_f##R(float* Kst, const ElasticConsts* ec, long P, hipStream_t);
PFDD_RED_DECL(1) PFDD_RED_DECL(2) PFDD_RED_DECL(3) PFDD_RED_DECL(4) PFDD_RED_DECL(5) PFDD_RED_DECL(6)
#undef PFDD_RED_DECL

}  // namespace pfdd
