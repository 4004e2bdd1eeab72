// Products of bf16 matrices with what stands around them in a layer of LoRA training.
#pragma once
#include <torch/extension.h>

// Columns of an output, as a sum of products a b: a (rows, k); b (width, k), or (k, width)
// where weights are taken as they lie in backward. No b: adds nothing.
struct ProductTerm {
  at::Tensor a;
  c10::optional<at::Tensor> b;
};
struct ProductBlock {
  int64_t width;
  std::vector<ProductTerm> terms;
  c10::optional<at::Tensor> bias;
};

// Whether the products below take these operands, whatever they hold yet: what a term is
// made of need not be launched for one that is refused. What they write is not asked for.
bool product_takes(const std::vector<ProductBlock>& blocks, bool rows_of_b);

// out <- the blocks side by side (+ res, clear of out): fp32 sums, rounded once.
// rows_of_b: b is (k, width). tile: the shape of tile, for tests; 0 picks one. All of
// them: false, and nothing done, for what 16 B accesses and steps of 32 of K can't walk.
bool product(const std::vector<ProductBlock>& blocks, bool rows_of_b, const at::Tensor& out,
             const c10::optional<at::Tensor>& res = {}, int tile = 0);

// gu, if wanted, <- [gate | up], act <- silu(gate) * up of both rounded; the terms of
// both have the same a, one for one
bool product_glu(const ProductBlock& gate, const ProductBlock& up,
                 const c10::optional<at::Tensor>& gu, const at::Tensor& act, int tile = 0);

// dgate, dup <- the activation's gradients for dact = the block, b (k, width); gu clear
// of both
bool product_glu_bwd(const ProductBlock& block, const at::Tensor& gu, const at::Tensor& dgate,
                     const at::Tensor& dup, int tile = 0);
