// The factorisation step of small ranks (fused.hip).
#pragma once

#include "dnpeff_internal.hpp"

namespace dn {

constexpr int FUSED_MAX_RANK = 64;
constexpr int64_t FU_CHUNKS = 4096;  // workgroups that A H^T is cut into where its rows allow

bool fused_supported(int64_t n, int64_t m, int64_t nnz, int r);
// What the lists and a context's buffers take at most.
double fused_bytes(int64_t n, int64_t nnz, int r);
// Tiles, packed entries and chunks of a matrix without dense head (needs csr_ensure_products).
int fused_plan_build(dnpeff_csr* S, int r);

// What a context keeps between the launches of a step.
struct fused_state {
  enum gram_state { NONE, PARTS, SUMMED };
  int r = 0, S_floats = 0, h_wgs = 0, w_wgs = 0;
  float* gh_part = nullptr;  // partial H^T H of the last H update, one per workgroup
  float* gw_part = nullptr;
  float* gh_sum = nullptr;
  float* gw_sum = nullptr;
  float* n_part = nullptr;   // A H^T by chunks
  int64_t n_part_floats = 0;
  double* dots = nullptr;
  gram_state gh_state = NONE, gw_state = NONE;

  int create(const dnpeff_csr* S, int64_t n, int rank);
  void destroy();
  int set_gram(const float* G, bool of_h);
  int product_n(const dnpeff_csr* S, const float* H);
  int sum_h();
  int sum_w();
  // Nw: A H^T [n, r], or NULL for the chunk sums of product_n
  int update_w(const dnpeff_csr* S, int64_t n, const float* Nw, float* W, float eps);
  int update_h(const dnpeff_csr* S, const float* W, float* H, float eps);
  // out2 (device or pinned) = <A H^T, W>, <W^T W, H^T H>
  int loss_sums(const dnpeff_csr* S, int64_t n, const float* Nw, const float* W, double* out2);
};

}  // namespace dn
