// 2DIR through one-exciton basis vectors (twodir_basis.hip), called by
// nise_2dir_batched after its checks.
#pragma once

#include <vector>

#include "nise_internal.h"

namespace nise {

struct BasisCall {
  const t_non *non;
  FrameSource src;
  std::vector<uint8_t> mask;  // union of kept couplings over the strict upper triangle
  std::vector<uint32_t> lex;  // the same as a | b << 16, lexicographic
  int end, do_gb, do_se, do_ea, es;
  int64_t f_lo, f_hi;
  const float *mu_rec;
  int64_t mu_stride;          // 0: static dipoles
  const float *anh_rec, *over_rec;
  hipStream_t st;
};
bool basis_path(const t_non *non, int K2, bool do_ea);
int run_basis(const BasisCall &c, float *R12);

}  // namespace nise
