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
