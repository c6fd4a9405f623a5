// pfdd_reduced.hip -- instantiations of the reduced-basis kernels.  Compiled
// with -DPFDD_RED_R=1..6 and -DPFDD_RED_KIND=0..3 (row kernel on the FP64,
// compensated or lean master; column kernels), once with KIND 4 (N2 pass) and with
// KIND 5 and 6 (plane kernel, FP64 and FP32).
#include <type_traits>

#include "pfdd_reduced.hpp"

namespace pfdd {
namespace {

#if PFDD_RED_KIND < 4
constexpr int R = PFDD_RED_R;
#endif

#if PFDD_RED_KIND < 3
template <typename T, int N, typename M> void row(const RedRowLaunch<T>& q, M xi) {
  const dim3 grid(q.nblk, q.batch);
  const bool opt = q.o.mask || q.o.taupp || q.o.extra || q.o.project;
  if constexpr (red_unrolled(R) > 0) {
    if (q.a.S <= red_unrolled(R)) {
      const dim3 block(RowRed<T, N, R, red_ppt(sizeof(T) == 8, N, R)>::NT);
      if (opt)
        hipLaunchKernelGGL((k_row_red<T, N, R, M, true>), grid, block, 0, q.stream, q.W, xi, q.a, q.o, q.tw, q.partials,
                           q.step_ctr);
      else
        hipLaunchKernelGGL((k_row_red<T, N, R, M, false>), grid, block, 0, q.stream, q.W, xi, q.a, q.o, q.tw,
                           q.partials, q.step_ctr);
      return;
    }
  }
  const dim3 block(RowRed<T, N, R, 1>::NT);
  if (opt)
    hipLaunchKernelGGL((k_row_red_n<T, N, R, M, true>), grid, block, 0, q.stream, q.W, xi, q.a, q.o, q.tw, q.partials,
                       q.step_ctr);
  else
    hipLaunchKernelGGL((k_row_red_n<T, N, R, M, false>), grid, block, 0, q.stream, q.W, xi, q.a, q.o, q.tw, q.partials,
                       q.step_ctr);
}
template <typename T, typename M> bool row_any(const RedRowLaunch<T>& q, M xi, int n3) {
  switch (n3) {
#define PFDD_L(NN) case NN: row<T, NN>(q, xi); return true;
    PFDD_L(2) PFDD_L(3) PFDD_L(4) PFDD_L(6) PFDD_L(8) PFDD_L(12) PFDD_L(16) PFDD_L(24)
    PFDD_L(32) PFDD_L(48) PFDD_L(64) PFDD_L(96) PFDD_L(128) PFDD_L(192) PFDD_L(256) PFDD_L(384) PFDD_L(512)
#undef PFDD_L
    default: return false;
  }
}
#elif PFDD_RED_KIND == 3
template <typename T, int N> void col(const RedColLaunch<T>& q) {
  using K = ColRed<T, N, R>;
  const int blocks = (int)((q.P / N + K::TC - 1) / K::TC * q.batch);
  const dim3 grid((unsigned)(blocks + (q.fin.in ? 1 : 0)));
  if (q.Kst)
    hipLaunchKernelGGL((k_col_red<T, N, R, true>), grid, dim3(K::NT), K::LDS, q.stream, q.W, q.ec, q.Kst, q.P, blocks, q.tw,
                       q.fin);
  else
    hipLaunchKernelGGL((k_col_red<T, N, R, false>), grid, dim3(K::NT), K::LDS, q.stream, q.W, q.ec, q.Kst, q.P, blocks, q.tw,
                       q.fin);
}
// The LDS limit of the tiles wider than 64 KB.
template <typename T, int N> bool col_attr() {
  constexpr int L = (int)ColRed<T, N, R>::LDS;
  if constexpr (L <= 64 * 1024) return true;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_col_red<T, N, R, true>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, L) == hipSuccess &&
         hipFuncSetAttribute(reinterpret_cast<const void*>(&k_col_red<T, N, R, false>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, L) == hipSuccess;
}
template <typename T> void build(T* Kst, const ElasticConsts* ec, long P, hipStream_t st) {
  hipLaunchKernelGGL((k_build_K<T, R>), dim3((unsigned)((P + 255) / 256)), dim3(256), 0, st, Kst, ec, P);
}
template <typename T> bool col_any(const RedColLaunch<T>& q, int n1) {
  switch (n1) {
#define PFDD_L(NN) case NN: col<T, NN>(q); return true;
    PFDD_L(2) PFDD_L(3) PFDD_L(4) PFDD_L(6) PFDD_L(8) PFDD_L(12) PFDD_L(16) PFDD_L(24)
    PFDD_L(32) PFDD_L(48) PFDD_L(64) PFDD_L(96) PFDD_L(128) PFDD_L(192) PFDD_L(256) PFDD_L(384) PFDD_L(512)
#undef PFDD_L
    default: return false;
  }
}
#elif PFDD_RED_KIND == 4
template <typename T, int N> void pass2(const RedPass2Launch<T>& q) {
  constexpr int TILE = tile_cols<T, N, RED_RL>(), NT = cols_threads<T, N, RED_RL>(), NW = NT / 64 > 0 ? NT / 64 : 1;
  const int blocks = (int)(q.outer * ((q.inner + TILE - 1) / TILE));
  const int nfold = q.fold.in ? (q.fold.F * FOLD + NW - 1) / NW : 0;
  hipLaunchKernelGGL((k_pass2_red<T, N>), dim3((unsigned)(blocks + nfold)), dim3(NT), (cols_lds_bytes<T, N, RED_RL>()),
                     q.stream, q.W, (int)q.inner, blocks, (T)q.sign, q.tw, q.fold, nfold);
}
template <typename T> bool pass2_any(const RedPass2Launch<T>& q, int n2) {
  switch (n2) {
#define PFDD_L(NN) case NN: pass2<T, NN>(q); return true;
    PFDD_L(2) PFDD_L(3) PFDD_L(4) PFDD_L(6) PFDD_L(8) PFDD_L(12) PFDD_L(16) PFDD_L(24)
    PFDD_L(32) PFDD_L(48) PFDD_L(64) PFDD_L(96) PFDD_L(128) PFDD_L(192) PFDD_L(256) PFDD_L(384) PFDD_L(512)
#undef PFDD_L
    default: return false;
  }
}
template <int N> bool pass2_attr() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pass2_red<double, N>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)cols_lds_bytes<double, N, RED_RL>()) == hipSuccess &&
         hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pass2_red<float, N>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)cols_lds_bytes<float, N, RED_RL>()) == hipSuccess;
}
#else
using T = std::conditional_t<PFDD_RED_KIND == 5, double, float>;
template <int N1, int N2> bool plane(const RedPlaneLaunch<T>& q) {
  if constexpr (N1 * N2 <= PLANE_MAX_POINTS) {
    const bool d = sizeof(T) == 8;
    const int blocks = q.n3 * (int)q.batch;
    hipLaunchKernelGGL((k_plane_red<T, N1, N2>), dim3((unsigned)(blocks + (q.fin.in ? 1 : 0))),
                       dim3((unsigned)plane_threads(d, N1, N2, q.R)), plane_lds(d, N1, N2, q.R), q.stream, q.W, q.ec,
                       q.Kst, q.n3, q.R, blocks, q.tw1, q.tw2, q.fin);
    return true;
  }
  return false;
}
template <int N1> bool plane_n2(const RedPlaneLaunch<T>& q, int n2) {
  switch (n2) {
#define PFDD_L(NN) case NN: return plane<N1, NN>(q);
    PFDD_L(2) PFDD_L(3) PFDD_L(4) PFDD_L(6) PFDD_L(8) PFDD_L(12) PFDD_L(16) PFDD_L(24)
    PFDD_L(32) PFDD_L(48) PFDD_L(64) PFDD_L(96) PFDD_L(128) PFDD_L(192) PFDD_L(256) PFDD_L(384) PFDD_L(512)
#undef PFDD_L
    default: return false;
  }
}
bool plane_any(const RedPlaneLaunch<T>& q, int n1, int n2) {
  if (!plane_fits(sizeof(T) == 8, n1, n2, q.R)) return false;
  switch (n1) {
#define PFDD_L(NN) case NN: return plane_n2<NN>(q, n2);
    PFDD_L(2) PFDD_L(3) PFDD_L(4) PFDD_L(6) PFDD_L(8) PFDD_L(12) PFDD_L(16) PFDD_L(24)
    PFDD_L(32) PFDD_L(48) PFDD_L(64) PFDD_L(96) PFDD_L(128) PFDD_L(192) PFDD_L(256) PFDD_L(384) PFDD_L(512)
#undef PFDD_L
    default: return false;
  }
}
#endif

}  // namespace

#define PFDD_CAT2(a, b) a##b
#define PFDD_CAT(a, b) PFDD_CAT2(a, b)
#if PFDD_RED_KIND == 0
bool PFDD_CAT(red_row_d, PFDD_RED_R)(const RedRowLaunch<double>& q, Master<double> xi, int n3) { return row_any(q, xi, n3); }
#elif PFDD_RED_KIND == 1
bool PFDD_CAT(red_row_c, PFDD_RED_R)(const RedRowLaunch<float>& q, MasterF32C xi, int n3) { return row_any(q, xi, n3); }
#elif PFDD_RED_KIND == 2
bool PFDD_CAT(red_row_l, PFDD_RED_R)(const RedRowLaunch<float>& q, MasterF32L xi, int n3) { return row_any(q, xi, n3); }
#elif PFDD_RED_KIND == 3
bool PFDD_CAT(red_col_d, PFDD_RED_R)(const RedColLaunch<double>& q, int n1) { return col_any(q, n1); }
bool PFDD_CAT(red_col_f, PFDD_RED_R)(const RedColLaunch<float>& q, int n1) { return col_any(q, n1); }
bool PFDD_CAT(red_col_attr, PFDD_RED_R)(int n1) {
  return n1 != 512 || (col_attr<double, 512>() && col_attr<float, 512>());
}
void PFDD_CAT(red_build_d, PFDD_RED_R)(double* K, const ElasticConsts* ec, long P, hipStream_t st) { build(K, ec, P, st); }
void PFDD_CAT(red_build_f, PFDD_RED_R)(float* K, const ElasticConsts* ec, long P, hipStream_t st) { build(K, ec, P, st); }
#elif PFDD_RED_KIND == 4
bool red_pass2_d(const RedPass2Launch<double>& q, int n2) { return pass2_any(q, n2); }
bool red_pass2_f(const RedPass2Launch<float>& q, int n2) { return pass2_any(q, n2); }
bool red_pass2_attr(int n2) {
  switch (n2) {
#define PFDD_L(NN) case NN: return pass2_attr<NN>();
    PFDD_L(2) PFDD_L(3) PFDD_L(4) PFDD_L(6) PFDD_L(8) PFDD_L(12) PFDD_L(16) PFDD_L(24)
    PFDD_L(32) PFDD_L(48) PFDD_L(64) PFDD_L(96) PFDD_L(128) PFDD_L(192) PFDD_L(256) PFDD_L(384) PFDD_L(512)
#undef PFDD_L
    default: return false;
  }
}
#elif PFDD_RED_KIND == 5
bool red_plane_d(const RedPlaneLaunch<double>& q, int n1, int n2) { return plane_any(q, n1, n2); }
int plane_threads(bool fp64, int n1, int n2, int R) {
  const int l1 = n2 * R * make_plan(n1, plane_rl(fp64, n1)).tpp, l2 = n1 * R * make_plan(n2, RED_RL).tpp;
  const int pts = n1 * n2 < 256 ? 256 : n1 * n2 < 512 ? n1 * n2 : 512;  // at least four waves: one block adds all sums
  int t = l1 > l2 ? l1 : l2;
  t = t > pts ? t : pts;
  return (t + 63) / 64 * 64;
}
size_t plane_lds(bool fp64, int n1, int n2, int R) {
  return (fp64 ? sizeof(double2) : sizeof(float2)) * ((size_t)n2 * R * (n1 + 1) + n1 + n2);
}
bool plane_fits(bool fp64, int n1, int n2, int R) {
  return n1 * n2 <= PLANE_MAX_POINTS && plane_threads(fp64, n1, n2, R) <= plane_max_threads(fp64) &&
         plane_lds(fp64, n1, n2, R) <= 60 * 1024;  // with the sums' 512 bytes, what a launch may use without asking
}
#else
bool red_plane_f(const RedPlaneLaunch<float>& q, int n1, int n2) { return plane_any(q, n1, n2); }
#endif

}  // namespace pfdd
