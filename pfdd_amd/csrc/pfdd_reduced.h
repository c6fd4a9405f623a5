// pfdd_reduced.h -- launchers of the reduced-basis kernels (pfdd_reduced.hip,
// compiled once per component count R and kind so that the instantiations
// build in parallel).
#pragma once
#include "pfdd_reduced.hpp"

namespace pfdd {

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
  void red_build_d##R(double* Kst, const ElasticConsts* ec, long P, hipStream_t);  \
  void red_build_f##R(float* Kst, const ElasticConsts* ec, long P, hipStream_t);
PFDD_RED_DECL(1) PFDD_RED_DECL(2) PFDD_RED_DECL(3) PFDD_RED_DECL(4) PFDD_RED_DECL(5) PFDD_RED_DECL(6)
#undef PFDD_RED_DECL

}  // namespace pfdd
