// The launch sequences of the fused 4-bit LoRA layers (hackathon_amd/fused_proj.py, lora.py) as
// native host code: one call from Python runs a whole forward or backward of a projection group or
// of the MLP.
//
// A training pass over one MLP is 23 launches and 40 allocations. Driven from Python each launch
// cost about 12 us of interpreter (argument checks, a size query, allocations, a stream object,
// ctypes), more than most of these kernels run: at 4 x 512 tokens of the 0.5B shape the MLP's
// forward and backward took 540-720 us of host time around 290 us of kernels. Here a launch costs
// the HIP runtime's 2-3 us and an allocation 0.5.
//
// The functions do what the Python ones beside them did, in the same order on the same stream:
// every operand is the caller's or allocated here from torch's allocator, nothing is kept between
// calls, and every kernel goes through the C-ABI of include/qlora_gfx950.h, whose addresses the
// binding passes in (`bind`), so this module links against torch alone.
#include <ATen/ATen.h>
#include <torch/csrc/utils/pybind.h>

#include <string>
#include <vector>

#include "../../../include/qlora_gfx950.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = c10::optional<Tensor>;

namespace {

#define QL_ENTRIES(X)                                                                             \
  X(qlora_nf4_dequant) X(qlora_nf4_dequant_t) X(qlora_nf4_dequant_group)                          \
  X(qlora_nf4_dequant_t_group) X(qlora_lora_down) X(qlora_lora_down_workspace_size)               \
  X(qlora_lora_dropout_down) X(qlora_lora_dropout_down_workspace_size) X(qlora_gemm_nt_cat)       \
  X(qlora_gemm_nt_cat_residual) X(qlora_gemm_nt_cat_workspace_size)                               \
  X(qlora_lora_up_masked_add_slots) X(qlora_lora_wgrad) X(qlora_lora_wgrad_workspace_size)        \
  X(qlora_lora_wgrad_diag) X(qlora_lora_wgrad_diag_workspace_size) X(qlora_lora_wgrad_masked)     \
  X(qlora_swiglu_fwd_lora_down) X(qlora_swiglu_fwd_lora_down_workspace_size)                      \
  X(qlora_swiglu_fwd_lora_down_dropout) X(qlora_swiglu_bwd_lora)                                  \
  X(qlora_swiglu_bwd_lora_workspace_size) X(qlora_swiglu_bwd_lora_dropout) X(qlora_strerror)

struct Entries {
#define QL_FIELD(name) decltype(&::name) name = nullptr;
  QL_ENTRIES(QL_FIELD)
#undef QL_FIELD
};
Entries ql;

std::vector<std::string> entry_names() {
  return {
#define QL_NAME(name) #name,
      QL_ENTRIES(QL_NAME)
#undef QL_NAME
  };
}

void bind(const std::vector<uint64_t>& addresses) {
  size_t i = 0;
  TORCH_CHECK(addresses.size() == entry_names().size(), "one address per entry point");
#define QL_SET(name) ql.name = reinterpret_cast<decltype(&::name)>(addresses[i++]);
  QL_ENTRIES(QL_SET)
#undef QL_SET
}

void check(int status, const char* what) {
  TORCH_CHECK(status == 0, what, " failed with status ", status, ": ", ql.qlora_strerror(status));
}
#define QL_CALL(name, ...) check(ql.name(__VA_ARGS__), #name)

constexpr int64_t kPad = 64;       // padded LoRA K segment: up to 4 adapters of rank 16
constexpr int64_t kNarrow = 2048;  // projections narrower than this share a forward GEMM

int tag(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return QL_F32;
    case at::kHalf: return QL_F16;
    case at::kBFloat16: return QL_BF16;
    default: TORCH_CHECK(false, "unsupported dtype ", t.scalar_type());
  }
}

// What the C-ABI's dtype tag and row stride describe: a 2-D matrix on a GPU, unit stride along
// its rows, of the given type.
void rows(const Tensor& t, at::ScalarType dtype, const char* name) {
  TORCH_CHECK_VALUE(t.is_cuda(), name, " must be on a GPU device");
  TORCH_CHECK_TYPE(t.scalar_type() == dtype, name, " is ", t.scalar_type(), "; this call takes ",
                   dtype, " operands");
  TORCH_CHECK_VALUE(t.dim() == 2 && (t.size(1) <= 1 || t.stride(1) == 1), name,
                    " must be a 2-D matrix with unit stride along its rows");
}

// Such a matrix of at least r x c, what the kernels read of it.
void matrix(const Tensor& t, at::ScalarType dtype, int64_t r, int64_t c, const char* name) {
  rows(t, dtype, name);
  TORCH_CHECK_VALUE(t.size(0) >= r && t.size(1) >= c, name, " is [", t.size(0), ", ", t.size(1),
                    "]; this call reads [", r, ", ", c, "]");
}

// A GEMM's bias: n consecutive values.
void vec(const Tensor& t, at::ScalarType dtype, int64_t n, const char* name) {
  TORCH_CHECK_VALUE(t.is_cuda(), name, " must be on a GPU device");
  TORCH_CHECK_TYPE(t.scalar_type() == dtype, name, " is ", t.scalar_type(), "; this call takes ",
                   dtype, " operands");
  TORCH_CHECK_VALUE(t.numel() == n && t.is_contiguous(), name, " must be ", n,
                    " consecutive values");
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }
bool pow2(int64_t v) { return v > 0 && (v & (v - 1)) == 0; }

// Columns [c0, c1) of a matrix, without a tensor for them.
struct Mat {
  char* p;
  int64_t ld, r, c;
};
Mat mat(const Tensor& t) {
  return {static_cast<char*>(t.data_ptr()), t.stride(0), t.size(0), t.size(1)};
}
Mat cols16(const Tensor& t, int64_t c0, int64_t c1) {
  Mat m = mat(t);
  m.p += 2 * c0;
  m.c = c1 - c0;
  return m;
}
Mat rows16(const Tensor& t, int64_t r0, int64_t r1) {
  Mat m = mat(t);
  m.p += 2 * r0 * m.ld;
  m.r = r1 - r0;
  return m;
}

struct Ctx {
  at::TensorOptions opts;  // the compute dtype on the device
  int dt;
  ql_stream_t stream;
  const float* table;      // the NF4 levels

  Ctx(const Tensor& like, uint64_t s, const Tensor& nf4_table)
      : opts(like.options().requires_grad(false)),
        dt(tag(like)),
        stream(reinterpret_cast<ql_stream_t>(s)),
        table(nf4_table.data_ptr<float>()) {}
  Tensor empty(int64_t r, int64_t c) const { return at::empty({r, c}, opts); }
  Tensor f32(int64_t r, int64_t c) const { return at::empty({r, c}, opts.dtype(at::kFloat)); }
  // [r, m] with a row stride that is a multiple of 8 (the transposed LoRA operands)
  Tensor t_buffer(int64_t r, int64_t m) const {
    return at::empty({r, (m + 7) / 8 * 8}, opts).narrow(1, 0, m);
  }
  Tensor workspace(int64_t bytes) const {
    return bytes > 0 ? at::empty({(bytes + 3) / 4}, opts.dtype(at::kFloat)) : Tensor();
  }
};
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// One NF4 weight: (packed, absmax, nested, code2, absmax2, offset, blocksize, blocksize2, rows,
// cols), the tensors kept alive by the caller's tuple.
struct Weight {
  Tensor packed, absmax, code2, absmax2;
  int nested;
  float offset;
  int bs, bs2;
  int64_t n, k;

  ql_nf4_weight desc(void* out) const {
    return {static_cast<const uint8_t*>(packed.data_ptr()), n, k, absmax.data_ptr(),
            static_cast<const float*>(ptr(code2)), static_cast<const float*>(ptr(absmax2)),
            offset, bs, bs2, out};
  }
};
Weight weight(const py::handle& h) {
  const auto t = h.cast<py::tuple>();
  Weight w;
  w.packed = t[0].cast<Tensor>();
  w.absmax = t[1].cast<Tensor>();
  w.nested = t[2].cast<int>();
  if (!t[3].is_none()) w.code2 = t[3].cast<Tensor>();
  if (!t[4].is_none()) w.absmax2 = t[4].cast<Tensor>();
  w.offset = t[5].cast<float>();
  w.bs = t[6].cast<int>();
  w.bs2 = t[7].cast<int>();
  w.n = t[8].cast<int64_t>();
  w.k = t[9].cast<int64_t>();
  TORCH_CHECK_VALUE(w.packed.is_cuda(), "HIP kernels need tensors on a GPU device");
  // two weights a byte, whatever type the bytes are stored as
  TORCH_CHECK_VALUE(w.packed.is_contiguous() && (int64_t)w.packed.nbytes() * 2 >= w.n * w.k,
                    "packed buffer is smaller than the quantised shape");
  return w;
}
std::vector<Weight> weights(const py::sequence& s) {
  std::vector<Weight> out;
  for (const auto& h : s) out.push_back(weight(h));
  return out;
}

// Every W_g [n_g, K] into its rows of w (one launch for up to 4 weights that the group kernel
// takes, else one each; a lone weight takes it for its stores, which stay in the caches).
void dequant(const Ctx& c, const std::vector<Weight>& ws, const Tensor& w) {
  ql_nf4_weight d[4];
  bool group = ws.size() >= 1 && ws.size() <= 4;
  int64_t off = 0;
  std::vector<char*> outs;
  for (const auto& x : ws) {
    TORCH_CHECK_VALUE(x.packed.numel() * 2 >= x.n * x.k,
                      "packed buffer is smaller than the quantised shape");
    char* out = static_cast<char*>(w.data_ptr()) + 2 * off * x.k;
    outs.push_back(out);
    off += x.n;
    group = group && x.nested == ws[0].nested && aligned(x.packed.data_ptr(), 4) &&
            aligned(out, 16) && pow2(x.bs) && x.bs >= 8 && (!x.nested || pow2(x.bs2)) &&
            x.n * x.k % 8 == 0;
  }
  if (group) {
    for (size_t i = 0; i < ws.size(); ++i) d[i] = ws[i].desc(outs[i]);
    QL_CALL(qlora_nf4_dequant_group, d, (int)ws.size(), ws[0].nested, c.table, c.dt, c.stream);
    return;
  }
  for (size_t i = 0; i < ws.size(); ++i) {
    const auto x = ws[i].desc(outs[i]);
    QL_CALL(qlora_nf4_dequant, x.packed, x.rows * x.cols, x.absmax, ws[i].nested, x.code2,
            x.absmax2, x.offset, x.blocksize, x.blocksize2, c.table, x.out, c.dt, c.stream);
  }
}

// Every W_g^T [K, n_g] into its columns of wt.
void dequant_t(const Ctx& c, const std::vector<Weight>& ws, const Tensor& wt) {
  ql_nf4_weight d[4];
  bool group = ws.size() >= 1 && ws.size() <= 4 && wt.stride(0) % 8 == 0;
  int64_t off = 0;
  std::vector<char*> outs;
  for (const auto& x : ws) {
    char* out = static_cast<char*>(wt.data_ptr()) + 2 * off;
    outs.push_back(out);
    off += x.n;
    group = group && x.nested == ws[0].nested && aligned(x.packed.data_ptr(), 16) &&
            aligned(out, 16) && pow2(x.bs) && x.bs >= 16 && (!x.nested || pow2(x.bs2)) &&
            x.k % 128 == 0 && x.n % 8 == 0;
  }
  if (group) {
    for (size_t i = 0; i < ws.size(); ++i) d[i] = ws[i].desc(outs[i]);
    QL_CALL(qlora_nf4_dequant_t_group, d, (int)ws.size(), ws[0].nested, c.table, wt.stride(0),
            c.dt, c.stream);
    return;
  }
  for (size_t i = 0; i < ws.size(); ++i) {
    const auto x = ws[i].desc(outs[i]);
    QL_CALL(qlora_nf4_dequant_t, x.packed, x.rows, x.cols, x.absmax, ws[i].nested, x.code2,
            x.absmax2, x.offset, x.blocksize, x.blocksize2, c.table, x.out, wt.stride(0), c.dt,
            c.stream);
  }
}

void lora_down(const Ctx& c, Mat x, Mat y, float alpha, Mat out, Mat out_t) {
  const int slots = (int)(y.r / 16);
  const int64_t bytes = ql.qlora_lora_down_workspace_size(x.r, x.c, slots);
  const Tensor ws = c.workspace(bytes);
  QL_CALL(qlora_lora_down, x.p, x.ld, y.p, y.ld, x.r, x.c, slots, c.dt, out.p, out.ld, (int)out.c,
          c.dt, alpha, out_t.p, out_t.ld, ptr(ws), bytes, c.stream);
}

// out = a b^T + a2 b2^T (+ bias) (+ residual); a2.p null: no second segment.
void gemm(const Ctx& c, Mat a, Mat b, Mat a2, Mat b2, Mat out, const Tensor& bias,
          const Tensor& residual) {
  const int64_t bytes = ql.qlora_gemm_nt_cat_workspace_size(a.r, b.r, a.c);
  const Tensor ws = c.workspace(bytes);
  const int64_t k2 = a2.p ? a2.c : 0;
  if (residual.defined()) {
    QL_CALL(qlora_gemm_nt_cat_residual, a.r, b.r, a.c, a.p, a.ld, b.p, b.ld, k2, a2.p, a2.ld, b2.p,
            b2.ld, c.dt, out.p, out.ld, c.dt, residual.data_ptr(), residual.stride(0), ptr(ws),
            bytes, c.stream);
  } else {
    QL_CALL(qlora_gemm_nt_cat, a.r, b.r, a.c, a.p, a.ld, b.p, b.ld, k2, a2.p, a2.ld, b2.p, b2.ld,
            c.dt, out.p, out.ld, c.dt, ptr(bias), 1.0f, ptr(ws), bytes, c.stream);
  }
}
const Mat kNone{nullptr, 0, 0, 0};

Tensor lora_wgrad(const Ctx& c, Mat pt, Mat q, float alpha, bool transposed) {
  const int slots = (int)(pt.r / 16);
  const Tensor out = transposed ? c.f32(pt.r, q.c) : c.f32(q.c, pt.r);
  const int64_t bytes = ql.qlora_lora_wgrad_workspace_size(q.r, q.c, slots);
  const Tensor ws = c.workspace(bytes);
  QL_CALL(qlora_lora_wgrad, pt.p, pt.ld, q.p, q.ld, q.r, q.c, slots, c.dt, out.data_ptr<float>(),
          (int)transposed, alpha, ptr(ws), bytes, c.stream);
  return out;
}

// The keep bits of G adapters' inputs [M, K].
void keep_bits(const std::vector<Tensor>& bits, int64_t G, int64_t M, int64_t K) {
  TORCH_CHECK_VALUE((int64_t)bits.size() == G, "one keep-bit tensor per adapter");
  for (const auto& b : bits) matrix(b, at::kByte, (M + 7) / 8, K, "bits");
}
std::vector<const uint8_t*> bit_ptrs(const std::vector<Tensor>& bits) {
  std::vector<const uint8_t*> p;
  for (const auto& b : bits) {
    TORCH_CHECK_VALUE(b.stride(0) == bits[0].stride(0), "the masks' bits must share one row stride");
    p.push_back(b.data_ptr<uint8_t>());
  }
  return p;
}

// The dropout state of a group: p = 0 for none, else A [16 G, K] and one mask per adapter.
struct Drop {
  double p = 0;
  Tensor a16;
  std::vector<Tensor> bits;
  float scale() const { return (float)(1.0 / (1.0 - p)); }
};

struct GroupForward {
  Tensor y, ut;
  std::vector<Tensor> bits;
};

// y [M, sum n_g] = x W_cat^T + u sB_cat^T + bias and u^T [16 G, M]; with p > 0 each adapter's u
// from its own dropout of x (Philox seed seeds[g]), its mask kept as bits.
GroupForward group_forward(const Ctx& c, const Tensor& x, const Tensor& a16, const Tensor& bs,
                           const std::vector<Weight>& ws, const Tensor& bias, double p,
                           const std::vector<uint64_t>& seeds) {
  const int64_t M = x.size(0), K = x.size(1), G = (int64_t)ws.size();
  int64_t N = 0;
  for (const auto& w : ws) {
    TORCH_CHECK_VALUE(w.k == K, "the weights take inputs of another width");
    N += w.n;
  }
  TORCH_CHECK_VALUE(a16.size(0) == 16 * G && a16.size(1) == K && bs.size(0) == N &&
                        bs.size(1) == kPad, "the packed adapters do not fit the group");
  if (bias.defined()) vec(bias, x.scalar_type(), N, "bias");
  GroupForward r;
  const Tensor u = c.empty(M, kPad);
  r.ut = c.t_buffer(16 * G, M);
  if (p > 0) {
    TORCH_CHECK_VALUE((int64_t)seeds.size() == G && K % 64 == 0, "one seed per adapter");
    Tensor xs = x;
    if (!aligned(x.data_ptr(), 16) || x.stride(0) % 8) xs = x.clone(at::MemoryFormat::Contiguous);
    std::vector<uint8_t*> bp;
    for (int64_t g = 0; g < G; ++g) {
      r.bits.push_back(at::empty({(M + 7) / 8, K}, c.opts.dtype(at::kByte)));
      bp.push_back(r.bits.back().data_ptr<uint8_t>());
    }
    const int64_t bytes = ql.qlora_lora_dropout_down_workspace_size(M, K, (int)G);
    const Tensor wk = c.workspace(bytes);
    QL_CALL(qlora_lora_dropout_down, xs.data_ptr(), xs.stride(0), a16.data_ptr(), a16.stride(0), M,
            K, (int)G, c.dt, seeds.data(), (float)p, (float)(1.0 / (1.0 - p)), nullptr, K,
            bp.data(), K, u.data_ptr(), u.stride(0), (int)kPad, r.ut.data_ptr(), r.ut.stride(0),
            ptr(wk), bytes, c.stream);
  } else {
    lora_down(c, mat(x), mat(a16), 1.0f, mat(u), mat(r.ut));
  }
  r.y = c.empty(M, N);
  const Tensor w = c.empty(N, K);
  dequant(c, ws, w);
  // a wide projection gets its own GEMM, narrow neighbours share one
  int64_t c0 = 0, width = 0;
  auto emit = [&](int64_t c1) {
    Tensor b = bias.defined() ? bias.view(-1).narrow(0, c0, c1 - c0) : Tensor();
    gemm(c, mat(x), rows16(w, c0, c1), mat(u), rows16(bs, c0, c1), cols16(r.y, c0, c1), b,
         Tensor());
    c0 = c1;
    width = 0;
  };
  int64_t off = 0;
  for (int64_t g = 0; g < G; ++g) {
    const int64_t n = ws[g].n;
    if (width > 0 && (width + n > kNarrow || n > kNarrow || width > kNarrow)) emit(off);
    off += n;
    width += n;
  }
  emit(off);
  return r;
}

struct GroupBackward {
  Tensor dx;
  std::vector<Tensor> ab;  // dA_0, dB_0, dA_1, ... (undefined where not needed)
};

// dx and the adapter gradients for the output gradient g [M, sum n_g]; du, dut: the adapters'
// down-projections of g when already made; db_given: the lora_B gradients when already made.
GroupBackward group_backward(const Ctx& c, const Tensor& g, const Tensor& x, const Tensor& at_pad,
                             const Tensor& bt, const Tensor& ut, const std::vector<Weight>& ws,
                             const std::vector<double>& scaling, bool need_dx,
                             const std::vector<bool>& need, Tensor du, Tensor dut,
                             const std::vector<Tensor>& db_given, const Drop& drop) {
  const int64_t M = g.size(0), K = x.size(1), G = (int64_t)ws.size();
  std::vector<int64_t> offs{0};
  for (const auto& w : ws) offs.push_back(offs.back() + w.n);
  const int64_t N = offs.back();
  TORCH_CHECK_VALUE(g.size(1) == N && x.size(0) == M && at_pad.size(0) == K && bt.size(1) == N &&
                        (int64_t)scaling.size() == G && (int64_t)need.size() == 2 * G,
                    "the group's operands do not fit together");
  const auto dt = x.scalar_type();
  matrix(bt, dt, 16 * G, N, "bt");
  matrix(ut, dt, 16 * G, M, "ut");
  TORCH_CHECK_VALUE(du.defined() == dut.defined(), "du and its transpose come together");
  if (du.defined()) {
    matrix(du, dt, M, 16 * G, "du");
    matrix(dut, dt, 16 * G, M, "dut");
  }
  matrix(at_pad, dt, K, du.defined() ? du.size(1) : kPad, "at");
  TORCH_CHECK_VALUE(db_given.empty() || (int64_t)db_given.size() == G,
                    "one lora_B gradient per adapter");
  if (drop.p > 0) {
    matrix(drop.a16, dt, 16 * G, K, "a16");
    keep_bits(drop.bits, G, M, K);
  }
  bool same = true;
  for (const double s : scaling) same = same && s == scaling[0];
  if (!du.defined()) {
    du = c.empty(M, kPad);
    dut = c.t_buffer(16 * G, M);
    if (same) {  // bt is block-diagonal: every adapter's du in one pass over g
      lora_down(c, mat(g), mat(bt), (float)scaling[0], mat(du), mat(dut));
    } else {
      for (int64_t i = 0; i < G; ++i) {
        Mat y = rows16(bt, 16 * i, 16 * i + 16);
        y.p += 2 * offs[i];
        y.c = ws[i].n;
        lora_down(c, cols16(g, offs[i], offs[i + 1]), y, (float)scaling[i],
                  cols16(du, 16 * i, kPad), rows16(dut, 16 * i, 16 * i + 16));
      }
    }
  }
  GroupBackward r;
  if (need_dx) {
    const Tensor wt = c.empty(K, N);
    dequant_t(c, ws, wt);
    r.dx = c.empty(M, K);
    if (drop.p == 0) {
      gemm(c, mat(g), mat(wt), mat(du), mat(at_pad), mat(r.dx), Tensor(), Tensor());
    } else {
      gemm(c, mat(g), mat(wt), kNone, kNone, mat(r.dx), Tensor(), Tensor());
      const auto bp = bit_ptrs(drop.bits);  // every adapter in one pass
      QL_CALL(qlora_lora_up_masked_add_slots, r.dx.data_ptr(), r.dx.stride(0), du.data_ptr(),
              du.stride(0), drop.a16.data_ptr(), drop.a16.stride(0), bp.data(),
              drop.bits[0].stride(0), (int)bp.size(), M, K, c.dt, drop.scale(), c.stream);
    }
  }
  bool need_a = false;
  int need_b = 0;
  for (int64_t i = 0; i < G; ++i) {
    need_a = need_a || need[2 * i];
    need_b += need[2 * i + 1];
  }
  Tensor da_all, db_all;
  if (need_a && drop.p > 0) {  // from x and the bits, every adapter in one pass over x
    const auto bp = bit_ptrs(drop.bits);
    da_all = c.f32(16 * G, K);
    const int64_t bytes = ql.qlora_lora_wgrad_workspace_size(M, K, (int)G);
    const Tensor wk = c.workspace(bytes);
    QL_CALL(qlora_lora_wgrad_masked, dut.data_ptr(), dut.stride(0), x.data_ptr(), x.stride(0), M,
            K, (int)G, c.dt, bp.data(), drop.bits[0].stride(0), drop.scale(),
            da_all.data_ptr<float>(), 1.0f, ptr(wk), bytes, c.stream);
  } else if (need_a) {
    da_all = lora_wgrad(c, mat(dut), mat(x), 1.0f, true);
  }
  if (db_given.empty() && need_b > 1) {  // every dB_g in one pass over g
    db_all = c.f32(N, 16);
    std::vector<float> al(scaling.begin(), scaling.end());
    const int64_t bytes = ql.qlora_lora_wgrad_diag_workspace_size(M, N, (int)G);
    const Tensor wk = c.workspace(bytes);
    QL_CALL(qlora_lora_wgrad_diag, ut.data_ptr(), ut.stride(0), g.data_ptr(), g.stride(0), M, N,
            (int)G, c.dt, offs.data(), al.data(), db_all.data_ptr<float>(), ptr(wk), bytes,
            c.stream);
  }
  for (int64_t i = 0; i < G; ++i) {
    Tensor da, db;
    if (need[2 * i]) da = G == 1 ? da_all : da_all.narrow(0, 16 * i, 16);
    if (need[2 * i + 1]) {
      if (!db_given.empty()) db = db_given[i];
      else if (db_all.defined()) db = db_all.narrow(0, offs[i], ws[i].n);
      else db = lora_wgrad(c, rows16(ut, 16 * i, 16 * i + 16), cols16(g, offs[i], offs[i + 1]),
                           (float)scaling[i], false);
    }
    r.ab.push_back(da);
    r.ab.push_back(db);
  }
  return r;
}

// ---- the Python entry points -----------------------------------------------------------------
py::object opt(const Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

Drop drop_of(double p, const OptTensor& a16, const std::vector<Tensor>& bits) {
  Drop d;
  d.p = p;
  if (p > 0) {
    TORCH_CHECK_VALUE(a16.has_value() && !bits.empty(), "dropout needs A and the masks");
    d.a16 = *a16;
    d.bits = bits;
  }
  return d;
}

py::tuple py_group_forward(const Tensor& x, const Tensor& a16, const Tensor& bs,
                           const py::sequence& specs, const OptTensor& bias, double p,
                           const std::vector<uint64_t>& seeds, const Tensor& table,
                           uint64_t stream) {
  rows(x, x.scalar_type(), "x");
  rows(a16, x.scalar_type(), "a16");
  rows(bs, x.scalar_type(), "bs");
  const Ctx c(x, stream, table);
  const auto ws = weights(specs);
  GroupForward r;
  {
    py::gil_scoped_release nogil;
    r = group_forward(c, x, a16, bs, ws, bias.value_or(Tensor()), p, seeds);
  }
  return py::make_tuple(r.y, r.ut, r.bits);
}

py::tuple py_group_backward(const Tensor& g, const Tensor& x, const Tensor& at_pad,
                            const Tensor& bt, const Tensor& ut, const py::sequence& specs,
                            const std::vector<double>& scaling, bool need_dx,
                            const std::vector<bool>& need, const OptTensor& du,
                            const OptTensor& dut, const std::vector<Tensor>& db_given, double p,
                            const OptTensor& a16, const std::vector<Tensor>& bits,
                            const Tensor& table, uint64_t stream) {
  const auto dt = x.scalar_type();
  rows(g, dt, "g");
  rows(x, dt, "x");
  rows(at_pad, dt, "at");
  rows(bt, dt, "bt");
  rows(ut, dt, "ut");
  const Ctx c(x, stream, table);
  const auto ws = weights(specs);
  GroupBackward r;
  {
    py::gil_scoped_release nogil;
    r = group_backward(c, g, x, at_pad, bt, ut, ws, scaling, need_dx, need, du.value_or(Tensor()),
                       dut.value_or(Tensor()), db_given, drop_of(p, a16, bits));
  }
  py::list ab;
  for (const auto& t : r.ab) ab.append(opt(t));
  return py::make_tuple(opt(r.dx), ab);
}

// nf4.lora_few's operands for a weight [N, K]: checked, and their addresses (checked from Python
// they cost a tenth of a four-row call: 40.4 us against 36.4 without).
py::tuple py_few_rows_operands(const Tensor& x, const Tensor& packed, const Tensor& a,
                               const Tensor& b, const OptTensor& bias, int64_t N, int64_t K) {
  TORCH_CHECK_VALUE(x.dim() == 2 && x.size(1) == K, "x has ", x.dim() ? x.size(-1) : 0,
                    " columns, the weight ", K);
  TORCH_CHECK_VALUE(a.dim() == 2 && a.size(0) == 16 && a.size(1) == K && b.dim() == 2 &&
                        b.size(0) == N && b.size(1) == 16,
                    "the factors must be [16, ", K, "] and [", N, ", 16], got ", a.sizes(), " and ",
                    b.sizes());
  const auto dt = x.scalar_type();
  TORCH_CHECK_TYPE((dt == at::kBFloat16 || dt == at::kHalf) && a.scalar_type() == at::kFloat &&
                       b.scalar_type() == at::kFloat,
                   "x must be bf16 or fp16 and the factors fp32, got ", dt, ", ", a.scalar_type(),
                   ", ", b.scalar_type());
  TORCH_CHECK_VALUE(x.stride(1) == 1 && a.is_contiguous() && b.is_contiguous() &&
                        packed.is_contiguous(),
                    "x must have unit stride along its rows; the factors and the packed codes must "
                    "be contiguous");
  TORCH_CHECK_VALUE((int64_t)packed.nbytes() * 2 >= N * K,
                    "packed buffer is smaller than the quantised shape");
  TORCH_CHECK_VALUE(x.is_cuda() && packed.is_cuda() && a.is_cuda() && b.is_cuda(),
                    "HIP kernels need tensors on a GPU device");
  if (bias.has_value()) vec(*bias, dt, N, "bias");
  const auto at = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()); };
  return py::make_tuple(at(x), at(packed), at(a), at(b),
                        bias.has_value() ? py::object(py::int_(at(*bias))) : py::none());
}

// The MLP after the gate | up group: h = silu(gate) up (not kept), the down adapter's u and, with
// dropout, its mask of h; out = [h | u] [W_d | sB_d]^T + bias (+ residual).
py::tuple py_mlp_down(const Tensor& y, const Tensor& a16, const Tensor& bs, const py::tuple& spec,
                      const OptTensor& bias_, const OptTensor& residual_, double p, uint64_t seed,
                      const Tensor& table, uint64_t stream) {
  rows(y, y.scalar_type(), "y");
  rows(a16, y.scalar_type(), "a16");
  rows(bs, y.scalar_type(), "bs");
  const Ctx c(y, stream, table);
  const std::vector<Weight> wd{weight(spec)};
  Tensor out, ut, bits;
  {
    py::gil_scoped_release nogil;
    const int64_t M = y.size(0), n = wd[0].k, N = wd[0].n;
    TORCH_CHECK_VALUE(y.size(1) == 2 * n && a16.size(1) == n && bs.size(0) == N,
                      "the down projection does not fit gate and up");
    matrix(a16, y.scalar_type(), 16, n, "a16");
    matrix(bs, y.scalar_type(), N, kPad, "bs");
    if (bias_.has_value()) vec(*bias_, y.scalar_type(), N, "bias");
    if (residual_.has_value() && !bias_.has_value()) {  // the GEMM adds it: read as y's type
      const Tensor& t = *residual_;
      TORCH_CHECK_VALUE(t.is_cuda() && t.scalar_type() == y.scalar_type(),
                        "a residual takes no bias, alpha 1 and out's dtype");
      TORCH_CHECK_VALUE(t.dim() == 2 && t.size(0) == M && t.size(1) == N && t.stride(1) == 1,
                        "residual must be [", M, ", ", N, "] with unit column stride");
    }
    const Tensor h = c.empty(M, n), u = c.empty(M, kPad);
    ut = c.t_buffer(16, M);
    const Mat gate = cols16(y, 0, n), up = cols16(y, n, 2 * n);
    const int64_t bytes = ql.qlora_swiglu_fwd_lora_down_workspace_size(M, n);
    {
      const Tensor wk = c.workspace(bytes);
      if (p == 0) {
        QL_CALL(qlora_swiglu_fwd_lora_down, gate.p, gate.ld, up.p, up.ld, h.data_ptr(), h.stride(0),
                M, n, a16.data_ptr(), a16.stride(0), 1.0f, c.dt, u.data_ptr(), u.stride(0),
                (int)kPad, ut.data_ptr(), ut.stride(0), ptr(wk), bytes, c.stream);
      } else {
        bits = at::empty({(M + 7) / 8, n}, c.opts.dtype(at::kByte));
        QL_CALL(qlora_swiglu_fwd_lora_down_dropout, gate.p, gate.ld, up.p, up.ld, h.data_ptr(),
                h.stride(0), M, n, a16.data_ptr(), a16.stride(0), 1.0f, c.dt, u.data_ptr(),
                u.stride(0), (int)kPad, ut.data_ptr(), ut.stride(0), seed, (float)p,
                (float)(1.0 / (1.0 - p)), bits.data_ptr<uint8_t>(), bits.stride(0), ptr(wk), bytes,
                c.stream);
      }
    }
    out = c.empty(M, N);
    const Tensor w = c.empty(N, n), bias = bias_.value_or(Tensor());
    const Tensor res = residual_.value_or(Tensor());
    dequant(c, wd, w);
    const bool fused = res.defined() && !bias.defined();  // else torch adds it
    gemm(c, mat(h), mat(w), mat(u), mat(bs), mat(out), bias, fused ? res : Tensor());
    if (res.defined() && !fused) out = res + out;
  }
  return py::make_tuple(out, ut, opt(bits));
}

// The MLP's backward: dy [M, N] to dx and the six adapter gradients (A_gate, B_gate, A_up, B_up,
// A_down, B_down).
py::tuple py_mlp_backward(const Tensor& dy, const Tensor& x, const Tensor& y, const Tensor& at_pad,
                          const Tensor& bt, const Tensor& ut, const py::sequence& specs,
                          const std::vector<double>& scaling, double p, const OptTensor& a16,
                          const std::vector<Tensor>& bits, const Tensor& at_d, const Tensor& bt_d,
                          const Tensor& ut_d, const py::tuple& spec_d, double s_d, double p_d,
                          const OptTensor& a16_d, const OptTensor& bits_d, bool need_dx,
                          const std::vector<bool>& need, const Tensor& table, uint64_t stream) {
  const auto dt = x.scalar_type();
  rows(dy, dt, "dy");
  rows(x, dt, "x");
  rows(y, dt, "y");
  rows(ut, dt, "ut");
  rows(ut_d, dt, "ut_d");
  const Ctx c(x, stream, table);
  const auto ws = weights(specs);
  const std::vector<Weight> wd{weight(spec_d)};
  GroupBackward r;
  Tensor da_d, db_d;
  {
    py::gil_scoped_release nogil;
    const int64_t M = x.size(0), n = wd[0].k, N = wd[0].n;
    TORCH_CHECK_VALUE(dy.size(0) == M && dy.size(1) == N && y.size(1) == 2 * n && ws.size() == 2 &&
                          scaling.size() == 2 && need.size() == 6 && bt.size(1) == 2 * n,
                      "the MLP's operands do not fit together");
    const bool masked = bits_d.has_value();
    matrix(y, dt, M, 2 * n, "y");
    matrix(bt, dt, 32, 2 * n, "bt");
    matrix(ut, dt, 32, M, "ut");
    matrix(bt_d, dt, 16, N, "bt_d");
    matrix(ut_d, dt, 16, M, "ut_d");
    if (masked) {
      TORCH_CHECK_VALUE(a16_d.has_value(), "dropout needs the down adapter's A");
      matrix(*a16_d, dt, 16, n, "a16_d");
      keep_bits({*bits_d}, 1, M, n);
    } else {
      matrix(at_d, dt, n, kPad, "at_d");
    }
    Tensor du_d = c.empty(M, kPad);
    const Tensor dut_d = c.t_buffer(16, M);
    // the SwiGLU kernel takes one row stride for all three (a saved-tensor hook may have packed
    // the forward's anew)
    TORCH_CHECK_VALUE(ut.stride(0) == dut_d.stride(0) && ut_d.stride(0) == dut_d.stride(0),
                      "ut, ut_d and du_d^T must share a row stride");
    lora_down(c, mat(dy), mat(bt_d), (float)s_d, mat(du_d), mat(dut_d));
    Tensor dh = c.empty(M, n);
    {
      const Tensor wt = c.empty(n, N);
      dequant_t(c, wd, wt);
      // with dropout the adapter term goes through its mask of h inside the SwiGLU backward
      gemm(c, mat(dy), mat(wt), masked ? kNone : mat(du_d), masked ? kNone : mat(at_d), mat(dh),
           Tensor(), Tensor());
    }
    if (need[5]) db_d = lora_wgrad(c, mat(ut_d), mat(dy), (float)s_d, false);
    const Tensor g = c.empty(M, 2 * n), du = c.empty(M, kPad), dut = c.t_buffer(32, M);
    const Tensor db_g = c.f32(n, 16), db_u = c.f32(n, 16);
    da_d = c.f32(16, n);
    const int64_t bytes = ql.qlora_swiglu_bwd_lora_workspace_size(M, n, 1);
    {
      const Tensor wk = c.workspace(bytes);
      const Mat gate = cols16(y, 0, n), up = cols16(y, n, 2 * n);
      const Mat dg = cols16(g, 0, n), dup = cols16(g, n, 2 * n);
      const Mat bt_g = rows16(bt, 0, 16);
      Mat bt_u = rows16(bt, 16, 32);
      bt_u.p += 2 * n;
      const Mat ut_g = rows16(ut, 0, 16), ut_u = rows16(ut, 16, 32);
      const float sg = (float)scaling[0], su = (float)scaling[1];
      if (!masked) {
        QL_CALL(qlora_swiglu_bwd_lora, dh.data_ptr(), dh.stride(0), gate.p, gate.ld, up.p, up.ld,
                dg.p, dg.ld, dup.p, dup.ld, M, n, bt_g.p, bt_u.p, bt_g.ld, ut_g.p, ut_u.p, ut_g.ld,
                sg, su, sg, su, c.dt, du.data_ptr(), du.stride(0), (int)kPad, dut.data_ptr(),
                dut.stride(0), db_g.data_ptr<float>(), db_u.data_ptr<float>(), dut_d.data_ptr(),
                1.0f, da_d.data_ptr<float>(), ptr(wk), bytes, c.stream);
      } else {
        QL_CALL(qlora_swiglu_bwd_lora_dropout, dh.data_ptr(), dh.stride(0), gate.p, gate.ld, up.p,
                up.ld, dg.p, dg.ld, dup.p, dup.ld, M, n, bt_g.p, bt_u.p, bt_g.ld, ut_g.p, ut_u.p,
                ut_g.ld, sg, su, sg, su, c.dt, du.data_ptr(), du.stride(0), (int)kPad,
                dut.data_ptr(), dut.stride(0), db_g.data_ptr<float>(), db_u.data_ptr<float>(),
                dut_d.data_ptr(), 1.0f, da_d.data_ptr<float>(), bits_d->data_ptr<uint8_t>(),
                bits_d->stride(0), (float)p_d, (float)(1.0 / (1.0 - p_d)), du_d.data_ptr(),
                du_d.stride(0), a16_d->data_ptr(), a16_d->stride(0), ptr(wk), bytes, c.stream);
      }
    }
    dh.reset();
    du_d.reset();
    r = group_backward(c, g, x, at_pad, bt, ut, ws, scaling, need_dx,
                       std::vector<bool>(need.begin(), need.begin() + 4), du, dut, {db_g, db_u},
                       drop_of(p, a16, bits));
  }
  py::list ab;
  for (const auto& t : r.ab) ab.append(opt(t));
  ab.append(need[4] ? opt(da_d) : py::none());
  ab.append(opt(db_d));
  return py::make_tuple(opt(r.dx), ab);
}

}  // namespace

PYBIND11_MODULE(_qlora_host, m) {
  // of the signatures it calls by address: compared with the kernel library's before binding
  m.attr("abi_version") = QLORA_ABI_VERSION;
  m.def("entry_names", &entry_names);
  m.def("bind", &bind);
  m.def("few_rows_operands", &py_few_rows_operands);
  m.def("group_forward", &py_group_forward);
  m.def("group_backward", &py_group_backward);
  m.def("mlp_down", &py_mlp_down);
  m.def("mlp_backward", &py_mlp_backward);
}
