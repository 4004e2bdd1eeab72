// Products of adapted projections that several sources share.
#pragma once
#include <torch/extension.h>

// out <- x m scaled, adapters m side by side: (r, K) each, or one (K, r); zeros in
// columns of out past the last one's.
struct AdapterInput {
  torch::Tensor x, out;
  std::vector<torch::Tensor> m;
  std::vector<double> scales;
};

// All of them in one launch. False, and nothing done, for ranks, strides or
// alignments that its 16 B accesses can't take.
bool adapter_inputs(const std::vector<AdapterInput>& jobs, bool k_major);

// act <- silu(gate) * up of gu = [gate | up], out <- scale * act m^T, m (r, F); zeros in
// columns of out past r. False, and nothing done, as above and for ranks past 64.
bool silu_mul_inputs(torch::Tensor gu, torch::Tensor act, torch::Tensor m, double scale,
                     torch::Tensor out);

// dgate, dup <- the activation's gradients for dact, out <- scaled dgate m[0] and dup m[1]
// side by side, m (F, r)
bool silu_mul_bwd_inputs(torch::Tensor dact, torch::Tensor gu, torch::Tensor dgate,
                         torch::Tensor dup, std::vector<torch::Tensor> m,
                         std::vector<double> scales, torch::Tensor out);
