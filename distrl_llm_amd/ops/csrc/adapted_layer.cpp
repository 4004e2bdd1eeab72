// The two halves of a decoder layer in LoRA training, each forward and backward as
// one call: attention and feed-forward with their norms, adapted projections and
// residual sums. The autograd nodes around them are models/fused_layer.py.
//
// An adapter is more of its projection: with u = scale * x A^T a projection is one
// sum, x W^T + u B^T, with its bias or the residual; backward is dY W + du A. Own
// products (product.hip) take all of them from where they lie, the activation and its
// gradient with them. For the library, where it is the faster or ranks don't fit, u
// lies beside x in one matrix, [x | u], for one product with [W | B]; where ranks don't
// fit few rows take large weights as they lie.
//
// Native because short micro-batches wait for the host: prepared in Python a pass of
// the 0.5B model over three short samples took 25.0 ms, with the library's products
// (17 us of the host each) and what they need beside them 17.8, now 15.6 (medians of
// processes in turn; single ones now 11.8 to 18.7, of which 8.5 are the kernels').
#include "adapted.h"
#include "product.h"

using at::Tensor;
using Tensors = std::vector<Tensor>;
using Ints = std::vector<int64_t>;
using Optional = c10::optional<Tensor>;

Tensor rmsnorm_fwd(Tensor x, Tensor w, double eps);
Tensor rmsnorm_bwd(Tensor dy, Tensor x, Tensor w, double eps);
Tensor rmsnorm_bwd_add(Tensor dy, Tensor x, Tensor w, Tensor g, double eps);
void rmsnorm_fwd_into(Tensor x, Tensor w, double eps, Tensor out);
void rope_rows(Tensor q, Tensor k, Tensor positions, Tensor inv_freq);
Tensors flash_varlen_fwd(Tensor q, Tensor k, Tensor v, Tensor cu, int64_t max_len, double scale,
                         Optional into);
void flash_varlen_bwd(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor cu,
                      int64_t max_len, double scale, Tensor dq, Tensor dk, Tensor dv);
Tensors adapter_grads(Tensors y, Tensors p, Ints by_col);
Tensor adapted_weight(Tensors w, Tensors b, int64_t pad);
Tensor stack_transposed(Tensors w, Ints at, int64_t cols);
bool lora_join(Tensor y, Tensor u, Tensor m, Tensor out, Optional res);
void silu_mul_packed_into(Tensor gu, Tensor out);
void silu_mul_bwd_packed(Tensor dy, Tensor gu, Tensor dgate, Tensor dup);

namespace {

// every operand is bf16 already
struct NoAutocast {
  c10::impl::ExcludeDispatchKeyGuard guard{c10::DispatchKey::AutocastCUDA};
};

Tensor columns(const Tensor& t, int64_t from, int64_t n) { return t.narrow(1, from, n); }

// Rows from which 32 of them a workgroup fill the chip: the activation then carries its
// adapter inputs along. A feed-forward half forward and back with the library's
// products, apart -> along, us: 1.5B, 2048, 4096, 7000, 9000, 16384 rows 730, 1103, 1717,
// 2072, 3324 -> 763, 1111, 1676, 2070, 3213; 4B, 4096, 8192, 12000 1558, 2851, 3804 -> 1568,
// 2803, 3730.
constexpr int64_t FULL = 8192;

Tensor heads(const Tensor& t, int64_t head_dim) {
  return t.view({t.size(0), t.size(1) / head_dim, head_dim});
}

// Rows of so many columns, an odd number of 128 B apart: 18793 x 1536 x 8960 took 465
// us with rows of 141 x 128 B, 513 with 140, 596 with 140.5.
Tensor apart_rows(int64_t rows, int64_t cols, const at::TensorOptions& options) {
  return columns(at::empty({rows, ((cols + 63) / 64 | 1) * 64}, options), 0, cols);
}

// out <- scale * a b, the scale in the product's epilogue
void scaled_mm(const Tensor& a, const Tensor& b, double scale, Tensor out) {
  at::addmm_out(out, out, a, b, 0., scale);
}

// Adapters of projections that share an input, or of one: A (r, K), B (N, r).
struct Adapters {
  // Adapters of 96 columns and more re-read a wider A for every 32 rows: from this
  // many rows on the GPU is behind the host, and the library's product faster on it
  // (18793 x 1536: 19.5 us for 28.9; 4816: 19.4 for 10.6).
  static constexpr int64_t MANY = 8192;

  Tensors A, B;
  std::vector<double> scales;
  Ints ranks, at;           // at: first column of each among the inputs u
  int64_t sum = 0, pad;     // pad: the columns they get beside their input

  Adapters(Tensors a, Tensors b, std::vector<double> s)
      : A(std::move(a)), B(std::move(b)), scales(std::move(s)) {
    TORCH_CHECK(!A.empty() && A.size() == B.size() && A.size() == scales.size());
    for (const auto& t : A) {
      at.push_back(sum);
      ranks.push_back(t.size(0));
      sum += t.size(0);
    }
    pad = (sum + 7) / 8 * 8;
  }

  Tensor part(const Tensor& u, size_t i) const { return columns(u, at[i], ranks[i]); }

  void clear_spare(const Tensor& u) const {
    if (pad > sum) columns(u, sum, pad - sum).zero_();
  }

  // u <- the adapters' scaled inputs side by side, zeros in spare columns
  void down(const Tensor& x, const Tensor& u) const {
    if ((pad <= 64 || x.size(0) < MANY) && adapter_inputs({{x, u, A, scales}}, false)) return;
    if (std::equal(scales.begin() + 1, scales.end(), scales.begin())) {
      scaled_mm(x, (A.size() > 1 ? at::cat(A) : A[0]).t(), scales[0], columns(u, 0, sum));
    } else {
      for (size_t i = 0; i < A.size(); ++i) scaled_mm(x, A[i].t(), scales[i], part(u, i));
    }
    clear_spare(u);
  }

  // du <- the gradients of the adapters' inputs
  void up(const Tensors& dy, const Tensor& du) const {
    std::vector<AdapterInput> jobs;
    for (size_t i = 0; i < B.size(); ++i)
      jobs.push_back({dy[i], i + 1 < B.size() ? part(du, i) : columns(du, at[i], pad - at[i]),
                      {B[i]}, {scales[i]}});
    if (adapter_inputs(jobs, true)) return;
    for (size_t i = 0; i < B.size(); ++i) scaled_mm(dy[i], B[i], scales[i], part(du, i));
    clear_spare(du);
  }
};

// Whether rows that products of our own don't take (an adapter's rank is no multiple of
// 32) take weights (N, K) as they lie, each projection's product in fp32 and its adapter
// joined to that, rather than laid out beside the adapter for one library product.
// Laying out moves the weights twice whatever the rows; joining moves every row and
// launches more, which small models wait for. A pass of a model over 62, 276, 686,
// 1352, 2008, 3687 and 6708 rows, laid out -> as they lie, ms: 7B 37.3, 42.3, 52.4,
// 74.4, 95.4, 146, 253 -> 27.4, 33.6, 45.2, 68.6, 93.2, 147, 262; 4B 29.5, 36.4, 45.3,
// 59.7, 71.7, 99, 187 -> 26.7, 33.9, 42.2, 57.8, 70.2, 106, 201; the 1.5B's gate and
// up (27.5M) at 62, 686 and 2008 rows 18.4, 23.6, 34.3 -> 19.9, 25.1, 34.6.
// Own products, where they take the operands, are the faster: a layer of 64, 700, 1400
// and 2048 rows, as they lie -> own, us: 7B 858, 1488, 2192, 3080 -> 570, 1270, 2188,
// 2491; 4B 589, 878, 1222, 1579 -> 332, 734, 1061, 1610; a pass over 89, 506 and 1278
// rows, ms: 7B 27.9, 39.6, 70.3 -> 22.8, 35.6, 63.6; 4B 25.7, 36.6, 52.9 -> 23.5, 33.0, 50.4.
bool apart(int64_t rows, int64_t N, int64_t K) { return rows <= 2048 && N * K >= 32 << 20; }

// out <- y + u m (+ res), y fp32
void join(const Tensor& y, const Tensor& u, const Tensor& m, const Tensor& out,
          const Optional& res = {}) {
  if (lora_join(y, u, m, out, res)) return;
  at::addmm_out(const_cast<Tensor&>(y), y, u, m, at::kFloat);
  if (res) y.add_(*res);
  out.copy_(y);
}

// Whether a product of many rows with wide weights (N, K) is the library's: its tiles
// are the faster there, and what it needs beside them (weights laid out beside
// adapters, the residual's copy, the activation's passes) small against that. A layer
// of 18793 rows, us, own -> library with all of it: down 440 -> 390, the input gradient of
// gate and up 850 -> 800, gate, up and activation 1080 -> 1060, the activation's gradient
// 840 -> 820, its epilogue not hidden behind another tile's products; but q, k, v 127 ->
// 160, o 111 -> 122.
// On either side of the line a feed-forward half, own -> library: 7000 and 8192 rows
// 1.5B 1537, 1783 -> 1676, 1650, 7B (6000) 5246, 6673 -> 5414, 6596; 9000, 12000, 16384
// rows 0.5B 828, 1022, 1350 -> 830, 1099, 1327, 1.5B 1791, 2639, 3434 -> 2030, 2453,
// 3075, 4B 2943, 3707, 5160 -> 2961, 3583, 4926, 7B 7199, 9559, 12608 -> 6660, 9193, 11860.
// And by width an attention half, whose widest are 6144 and 4608: 9000 and 16384 rows
// 4B 1472, 2482 -> 1595, 2655, 7B 1495, 2637 -> 1502, 2766; the 0.5B's down (4864), with
// the rest of its half, 807, 1329 -> 830, 1327.
bool library(int64_t rows, int64_t N, int64_t K) { return rows > 8192 && std::max(N, K) >= 8192; }

// x W^T + u B^T of projections of one input
std::vector<ProductBlock> blocks(const Tensor& x, const Tensor& u, const Tensors& W,
                                 const Adapters& ad, const std::vector<Optional>& bias) {
  std::vector<ProductBlock> out;
  for (size_t i = 0; i < W.size(); ++i)
    out.push_back({W[i].size(0), {{x, W[i]}, {ad.part(u, i), ad.B[i]}},
                   i < bias.size() ? bias[i] : Optional()});
  return out;
}

// the same of [x | u], + their biases, or + a residual: one rounding for all of it
Tensor projected(const Tensor& xu, const Tensors& W, const Adapters& ad,
                 const std::vector<Optional>& bias, const Optional& res = {}) {
  const int64_t rows = xu.size(0), K = W[0].size(1);
  int64_t width = 0;
  bool any = false;
  for (const auto& w : W) width += w.size(0);
  for (const auto& b : bias) any = any || b;
  if (!library(rows, width, K)) {
    const auto sums = blocks(columns(xu, 0, K), columns(xu, K, ad.pad), W, ad, bias);
    if (product_takes(sums, false)) {
      auto out = at::empty({rows, width}, xu.options());
      if (product(sums, false, out, res)) return out;
    }
  }
  if (apart(rows, width, K)) {
    auto out = at::empty({rows, width}, xu.options());
    const auto x = columns(xu, 0, K), u = columns(xu, K, ad.pad);
    int64_t from = 0;
    for (size_t i = 0; i < W.size(); ++i) {
      const int64_t n = W[i].size(0);
      join(at::mm(x, W[i].t(), at::kFloat), ad.part(u, i), ad.B[i].t(), columns(out, from, n),
           res ? res : any && bias[i] ? Optional(bias[i]->expand({rows, n})) : Optional());
      from += n;
    }
    return out;
  }
  const auto WB = adapted_weight(W, ad.B, ad.pad);
  if (res) return at::addmm(*res, xu, WB.t());
  if (!any) return at::mm(xu, WB.t());
  Tensors all;
  for (size_t i = 0; i < bias.size(); ++i)
    all.push_back(bias[i] ? *bias[i] : at::zeros({W[i].size(0)}, xu.options()));
  return at::addmm(at::cat(all), xu, WB.t());
}

// a b, from a long K, in runs of rows whose 256 x 256 tiles the chip has at once: past a
// full wave the library's product of all rows takes as long as for two, or picks another
// kernel (18793 x 17984 x 1536 1129 us, 16384 rows 671, 10752 rows, one wave, 384). What
// is left beyond half a wave is a full one too, over rows that are done already: the
// library takes 316 to 618 us for 5700 to 9400 rows of that product.
// Sums over 24 row counts of one to four waves, all rows at once -> in runs, ms: K 9792,
// 896 columns 4.07 -> 2.99; 6208, 1024 2.65 -> 2.59; 17984, 1536 24.8 -> 19.7 (two
// products of half K 24.7); 22080, 2048 40.0 -> 31.6; 19520, 2560 28.9 -> 22.4; 37952,
// 3584 67.7 -> 49.9; 28736, 4096 56.0 -> 41.1; 27712, 5120 48.9 -> 37.3; one row count
// alone 0.47 to 1.16 of its time.
Tensor in_waves(const Tensor& a, const Tensor& b) {
  const int64_t rows = a.size(0), cols = b.size(1);
  constexpr int64_t CUS = 256;
  const int64_t wave = std::max<int64_t>(1, CUS / ((cols + 255) / 256)) * 256;
  if (rows <= wave) return at::mm(a, b);
  auto out = at::empty({rows, cols}, a.options());
  for (int64_t done = 0; done < rows; done += wave) {
    const bool full = 2 * (rows - done) > wave;
    const int64_t from = full ? std::min(done, rows - wave) : done;
    const int64_t n = full ? wave : rows - done;
    auto part = out.narrow(0, from, n);
    at::mm_out(part, a.narrow(0, from, n), b);
  }
  return out;
}

// dY W + du A of projections of one input, their W and A as they lie
Tensor back_apart(const Tensors& dy, const Tensors& W, const Tensor& du, const Adapters& ad) {
  auto y = at::mm(dy[0], W[0], at::kFloat);
  for (size_t i = 1; i < W.size(); ++i) at::addmm_out(y, y, dy[i], W[i], at::kFloat);
  auto out = at::empty(y.sizes(), dy[0].options());
  join(y, columns(du, 0, ad.sum), ad.A.size() > 1 ? at::cat(ad.A) : ad.A[0], out);
  return out;
}

struct Through { Tensor dx, du; };

// g W + du A with du = scale * g B, and du
Through through(const Tensor& g, const Tensor& W, const Adapters& ad) {
  const int64_t N = g.size(1);
  if (!library(g.size(0), N, W.size(1))) {
    auto du = at::empty({g.size(0), ad.pad}, g.options());
    const auto r = ad.part(du, 0);
    const std::vector<ProductBlock> sum{{W.size(1), {{g, W}, {r, ad.A[0]}}, {}}};
    if (product_takes(sum, true)) {
      auto dx = at::empty({g.size(0), W.size(1)}, g.options());
      ad.up({g}, du);
      if (product(sum, true, dx)) return {dx, r};
    }
  }
  if (apart(g.size(0), N, W.size(1))) {
    auto du = at::empty({g.size(0), ad.pad}, g.options());
    ad.up({g}, du);
    return {back_apart({g}, {W}, du, ad), ad.part(du, 0)};
  }
  auto gd = at::empty({g.size(0), N + ad.pad}, g.options());
  auto g2 = columns(gd, 0, N), du = columns(gd, N, ad.pad);
  g2.copy_(g);
  ad.up({g}, du);
  return {at::mm(gd, stack_transposed({W, ad.A[0]}, {0, N}, N + ad.pad).t()), ad.part(du, 0)};
}

// dx <- dY W + du A of projections of one input; false where that is the library's
bool own_dx(Tensor& dx, const Tensors& W, const Tensors& dy, const Tensor& du, const Adapters& ad) {
  const int64_t rows = du.size(0);
  ProductBlock sum{W[0].size(1), {}, {}};
  int64_t K = 0;
  for (size_t i = 0; i < W.size(); ++i) {
    sum.terms.push_back({dy[i], W[i]});
    K += W[i].size(0);
  }
  if (library(rows, sum.width, K)) return false;
  for (size_t i = 0; i < W.size(); ++i) sum.terms.push_back({ad.part(du, i), ad.A[i]});
  if (!product_takes({sum}, true)) return false;
  dx = at::empty({rows, sum.width}, du.options());
  return product({sum}, true, dx);
}

struct Job { Tensor y, p; bool by_col; };

// p^T y of every job over the rows: gradients of A, or of B (by_col, transposed).
// Ranks that the kernel does not take go through the library.
Tensors sums(const std::vector<Job>& jobs) {
  Tensors out(jobs.size()), y, p;
  Ints by_col, own;
  for (size_t i = 0; i < jobs.size(); ++i) {
    const auto& j = jobs[i];
    const int64_t r = j.p.size(1);
    if (r % 8 == 0 && r >= 8 && r <= 128 && j.y.size(1) % 8 == 0 && j.p.size(0) > 0) {
      own.push_back(i);
      y.push_back(j.y);
      p.push_back(j.p);
      by_col.push_back(j.by_col);
    } else {
      out[i] = j.by_col ? at::mm(j.y.t(), j.p) : at::mm(j.p.t(), j.y);
    }
  }
  if (!own.empty()) {
    auto got = adapter_grads(y, p, by_col);
    for (size_t i = 0; i < own.size(); ++i) out[own[i]] = got[i];
  }
  return out;
}

// gradients of the adapters in the order of their parameters: A, B of each
Tensors in_order(const Adapters& ad, const Tensor& dA, const Tensor* dB) {
  Tensors out;
  for (size_t i = 0; i < ad.A.size(); ++i) {
    out.push_back(dA.narrow(0, ad.at[i], ad.ranks[i]));
    out.push_back(dB[i]);
  }
  return out;
}

}  // namespace

// y = x + o_proj(attention(qkv_proj(norm(x)))) over rows x of sequences that begin
// at cu. W, A, B, scales: q, k, v, o. Returns y and what backward needs:
// [x | u] of the projections, [attention | u] of o, q, k, v, lse and, with head
// norms, q and k before them.
Tensors attention_half_fwd(Tensor x, Tensor norm, double eps, Tensors W,
                           std::vector<Optional> bias, Tensors A, Tensors B,
                           std::vector<double> scales, Optional q_norm, Optional k_norm,
                           double q_eps, double k_eps, Tensor pos, Tensor inv_freq, Tensor cu,
                           int64_t longest, double scale, int64_t head_dim) {
  NoAutocast plain;
  TORCH_CHECK(W.size() == 4 && A.size() == 4 && B.size() == 4 && scales.size() == 4 &&
              bias.size() == 3 && q_norm.has_value() == k_norm.has_value());
  const int64_t rows = x.size(0), hidden = x.size(1);
  const Adapters in({A[0], A[1], A[2]}, {B[0], B[1], B[2]}, {scales[0], scales[1], scales[2]});
  const Adapters o_ad({A[3]}, {B[3]}, {scales[3]});
  const Ints sizes = {W[0].size(0), W[1].size(0), W[2].size(0)};

  auto hu = apart_rows(rows, hidden + in.pad, x.options());
  auto h = columns(hu, 0, hidden);
  rmsnorm_fwd_into(x, norm, eps, h);
  in.down(h, columns(hu, hidden, in.pad));
  auto qkv = projected(hu, {W[0], W[1], W[2]}, in, bias);
  auto q = heads(columns(qkv, 0, sizes[0]), head_dim);
  auto k = heads(columns(qkv, sizes[0], sizes[1]), head_dim);
  auto v = heads(columns(qkv, sizes[0] + sizes[1], sizes[2]), head_dim);
  Tensor q0, k0;
  if (q_norm) {
    q0 = q.contiguous();
    k0 = k.contiguous();
    q = rmsnorm_fwd(q0, *q_norm, q_eps);
    k = rmsnorm_fwd(k0, *k_norm, k_eps);
  }
  rope_rows(q, k, pos, inv_freq);
  auto ou = apart_rows(rows, sizes[0] + o_ad.pad, x.options());
  auto o = columns(ou, 0, sizes[0]);
  auto lse = flash_varlen_fwd(q, k, v, cu, longest, scale, heads(o, head_dim))[1];
  o_ad.down(o, columns(ou, sizes[0], o_ad.pad));
  auto y = projected(ou, {W[3]}, o_ad, {}, x);
  return {y, hu, ou, q, k, v, lse, q0, k0};
}

// dx (undefined unless wanted), then the gradients of A and B of q, k, v, o.
Tensors attention_half_bwd(Tensor g, Tensor x, Tensor norm, double eps, Tensors W, Tensors A,
                           Tensors B, std::vector<double> scales, Optional q_norm,
                           Optional k_norm, double q_eps, double k_eps, Tensor pos,
                           Tensor back_freq, Tensor cu, int64_t longest, double scale, Tensor hu,
                           Tensor ou, Tensor q, Tensor k, Tensor v, Tensor lse, Optional q0,
                           Optional k0, bool want_dx) {
  NoAutocast plain;
  const int64_t rows = x.size(0), hidden = x.size(1), head_dim = q.size(2);
  const Adapters in({A[0], A[1], A[2]}, {B[0], B[1], B[2]}, {scales[0], scales[1], scales[2]});
  const Adapters o_ad({A[3]}, {B[3]}, {scales[3]});
  const Ints sizes = {W[0].size(0), W[1].size(0), W[2].size(0)};
  const int64_t width = sizes[0] + sizes[1] + sizes[2];
  g = g.contiguous();
  auto h = columns(hu, 0, hidden), u = columns(hu, hidden, in.pad);
  auto o = columns(ou, 0, sizes[0]), uo = columns(ou, sizes[0], o_ad.ranks[0]);

  const auto [dO, duo] = through(g, W[3], o_ad);
  auto dyu = at::empty({rows, width + in.pad}, x.options());
  const Tensors dys = {columns(dyu, 0, sizes[0]), columns(dyu, sizes[0], sizes[1]),
                       columns(dyu, sizes[0] + sizes[1], sizes[2])};
  auto du = columns(dyu, width, in.pad);
  auto dq = heads(dys[0], head_dim), dk = heads(dys[1], head_dim), dv = heads(dys[2], head_dim);
  flash_varlen_bwd(heads(dO, head_dim), q, k, v, heads(o, head_dim), lse, cu, longest, scale, dq,
                   dk, dv);
  // a rotation's gradient is the rotation by the negative angle
  rope_rows(dq, dk, pos, back_freq);
  if (q0) {
    dq.copy_(rmsnorm_bwd(dq.contiguous(), *q0, *q_norm, q_eps));
    dk.copy_(rmsnorm_bwd(dk.contiguous(), *k0, *k_norm, k_eps));
  }
  in.up(dys, du);
  auto s = sums({{h, du, false},
                 {o, duo, false},
                 {g, uo, true},
                 {dys[0], in.part(u, 0), true},
                 {dys[1], in.part(u, 1), true},
                 {dys[2], in.part(u, 2), true}});
  Tensors out = in_order(in, s[0], &s[3]);
  out.push_back(s[1]);
  out.push_back(s[2]);
  Tensor dx;
  if (want_dx && own_dx(dx, {W[0], W[1], W[2]}, dys, du, in)) {
    dx = rmsnorm_bwd_add(dx, x, norm, g, eps);
  } else if (want_dx && apart(rows, width, hidden)) {
    dx = rmsnorm_bwd_add(back_apart(dys, {W[0], W[1], W[2]}, du, in), x, norm, g, eps);
  } else if (want_dx) {
    const auto WA = stack_transposed({W[0], W[1], W[2], A[0], A[1], A[2]},
                                     {0, sizes[0], sizes[0] + sizes[1], width, width + in.at[1],
                                      width + in.at[2]}, width + in.pad);
    dx = rmsnorm_bwd_add(at::mm(dyu, WA.t()), x, norm, g, eps);
  }
  out.insert(out.begin(), dx);
  return out;
}

// y = x + down_proj(silu(gate_proj(norm(x))) * up_proj(norm(x))) over rows x. W, A,
// B, scales: gate, up, down. Returns y, [x | u], [gate | up], [act | u].
Tensors feed_forward_half_fwd(Tensor x, Tensor norm, double eps, Tensors W,
                              std::vector<Optional> bias, Tensors A, Tensors B,
                              std::vector<double> scales) {
  NoAutocast plain;
  TORCH_CHECK(W.size() == 3 && A.size() == 3 && B.size() == 3 && scales.size() == 3 &&
              bias.size() == 2);
  const int64_t rows = x.size(0), hidden = x.size(1), inner = W[0].size(0);
  const Adapters in({A[0], A[1]}, {B[0], B[1]}, {scales[0], scales[1]});
  const Adapters d_ad({A[2]}, {B[2]}, {scales[2]});
  auto hu = apart_rows(rows, hidden + in.pad, x.options());
  auto h = columns(hu, 0, hidden);
  rmsnorm_fwd_into(x, norm, eps, h);
  in.down(h, columns(hu, hidden, in.pad));
  auto au = apart_rows(rows, inner + d_ad.pad, x.options());
  auto act = columns(au, 0, inner);
  Tensor gu;
  bool ready = false;                     // act's adapter inputs
  if (!library(rows, 2 * inner, hidden)) {
    const auto both = blocks(h, columns(hu, hidden, in.pad), {W[0], W[1]}, in, bias);
    const auto &ug = both[0].terms[1].a, &uu = both[1].terms[1].a;
    const ProductBlock gate{inner, {both[0].terms[0], {ug, B[0]}, {uu, {}}}, bias[0]};
    const ProductBlock up{inner, {both[1].terms[0], {ug, {}}, {uu, B[1]}}, bias[1]};
    if (product_takes({gate, up}, false)) {
      gu = at::empty({rows, 2 * inner}, x.options());
      if (!product_glu(gate, up, gu, act)) gu = Tensor();
    }
  }
  if (!gu.defined()) {
    gu = projected(hu, {W[0], W[1]}, in, bias);
    ready = rows >= FULL && silu_mul_inputs(gu, act, A[2], scales[2], columns(au, inner, d_ad.pad));
    if (!ready) silu_mul_packed_into(gu, act);
  }
  if (!ready) d_ad.down(act, columns(au, inner, d_ad.pad));
  auto y = projected(au, {W[2]}, d_ad, {}, x);
  return {y, hu, gu, au};
}

// dx (undefined unless wanted), then the gradients of A and B of gate, up, down.
Tensors feed_forward_half_bwd(Tensor g, Tensor x, Tensor norm, double eps, Tensors W, Tensors A,
                              Tensors B, std::vector<double> scales, Tensor hu, Tensor gu,
                              Tensor au, bool want_dx) {
  NoAutocast plain;
  const int64_t rows = x.size(0), hidden = x.size(1), inner = W[0].size(0);
  const Adapters in({A[0], A[1]}, {B[0], B[1]}, {scales[0], scales[1]});
  const Adapters d_ad({A[2]}, {B[2]}, {scales[2]});
  g = g.contiguous();
  auto h = columns(hu, 0, hidden), u = columns(hu, hidden, in.pad);
  auto act = columns(au, 0, inner), ud = columns(au, inner, d_ad.ranks[0]);

  auto dyu = apart_rows(rows, 2 * inner + in.pad, x.options());
  auto dgate = columns(dyu, 0, inner), dup = columns(dyu, inner, inner),
       du = columns(dyu, 2 * inner, in.pad);
  Tensor dud;
  bool ready = false;                     // dgate's and dup's adapter inputs
  if (!library(rows, hidden, inner)) {
    auto both = at::empty({rows, d_ad.pad}, x.options());
    const auto r = d_ad.part(both, 0);
    const ProductBlock dact{inner, {{g, W[2]}, {r, A[2]}}, {}};
    if (product_takes({dact}, true)) {
      d_ad.up({g}, both);
      if (product_glu_bwd(dact, gu, dgate, dup)) dud = r;
    }
  }
  if (!dud.defined()) {
    const auto [dact, du2] = through(g, W[2], d_ad);
    ready = rows >= FULL &&
            silu_mul_bwd_inputs(dact, gu, dgate, dup, {B[0], B[1]}, {scales[0], scales[1]}, du);
    if (!ready) silu_mul_bwd_packed(dact, gu, dgate, dup);
    dud = du2;
  }
  if (!ready) in.up({dgate, dup}, du);
  auto s = sums({{h, du, false},
                 {act, dud, false},
                 {g, ud, true},
                 {dgate, in.part(u, 0), true},
                 {dup, in.part(u, 1), true}});
  Tensors out = in_order(in, s[0], &s[3]);
  out.push_back(s[1]);
  out.push_back(s[2]);
  Tensor dx;
  if (want_dx && own_dx(dx, {W[0], W[1]}, {dgate, dup}, du, in)) {
    dx = rmsnorm_bwd_add(dx, x, norm, g, eps);
  } else if (want_dx && apart(rows, 2 * inner, hidden)) {
    dx = rmsnorm_bwd_add(back_apart({dgate, dup}, {W[0], W[1]}, du, in), x, norm, g, eps);
  } else if (want_dx) {
    const auto WA = stack_transposed({W[0], W[1], A[0], A[1]},
                                     {0, inner, 2 * inner, 2 * inner + in.ranks[0]},
                                     2 * inner + in.pad);
    dx = rmsnorm_bwd_add(in_waves(dyu, WA.t()), x, norm, g, eps);
  }
  out.insert(out.begin(), dx);
  return out;
}

namespace {

bool all_bf16(const Tensors& ts) {
  for (const auto& t : ts)
    if (!t.is_cuda() || t.scalar_type() != at::kBFloat16) return false;
  return true;
}

}  // namespace

// x W^T of projections of one input side by side, with their adapters (one each, or
// none at all) and biases, or + res, in one rounding. None where own products don't
// take the operands.
Optional adapted_projection(Tensor x, Tensors W, std::vector<Optional> bias, Tensors A, Tensors B,
                            std::vector<double> scales, Optional res) {
  if (!all_bf16(W) || !all_bf16(A) || !all_bf16(B) || !all_bf16({x}) || x.size(0) == 0) return {};
  int64_t width = 0;
  for (const auto& w : W) width += w.size(0);
  std::vector<ProductBlock> sums;
  if (A.empty()) {
    for (size_t i = 0; i < W.size(); ++i) sums.push_back({W[i].size(0), {{x, W[i]}}, bias.at(i)});
    if (!product_takes(sums, false)) return {};
  } else {
    TORCH_CHECK(A.size() == W.size());
    const Adapters ad(A, B, scales);
    const auto u = at::empty({x.size(0), ad.pad}, x.options());
    sums = blocks(x, u, W, ad, bias);
    if (!product_takes(sums, false)) return {};
    ad.down(x, u);
  }
  auto out = at::empty({x.size(0), width}, x.options());
  if (!product(sums, false, out, res)) return {};
  return out;
}

// silu(x Wg^T) * (x Wu^T), the same way
Optional adapted_activation(Tensor x, Tensors W, Tensors A, Tensors B, std::vector<double> scales) {
  if (!all_bf16(W) || !all_bf16(A) || !all_bf16(B) || !all_bf16({x}) || x.size(0) == 0) return {};
  TORCH_CHECK(W.size() == 2 && (A.empty() || A.size() == 2));
  const int64_t inner = W[0].size(0);
  ProductBlock gate{inner, {{x, W[0]}}, {}}, up{inner, {{x, W[1]}}, {}};
  if (A.empty()) {
    if (!product_takes({gate, up}, false)) return {};
  } else {
    const Adapters ad(A, B, scales);
    const auto u = at::empty({x.size(0), ad.pad}, x.options());
    const auto ug = ad.part(u, 0), uu = ad.part(u, 1);
    gate.terms.insert(gate.terms.end(), {{ug, B[0]}, {uu, {}}});
    up.terms.insert(up.terms.end(), {{ug, {}}, {uu, B[1]}});
    if (!product_takes({gate, up}, false)) return {};
    ad.down(x, u);
  }
  auto act = at::empty({x.size(0), inner}, x.options());
  if (!product_glu(gate, up, {}, act)) return {};
  return act;
}
