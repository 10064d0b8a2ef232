// Per-row cross-entropy statistics over a chunk of logits, with the in-place gradient,
// for gfx950.
//
// Reference semantics: solution/fused_ce.py:42-96 (ce_row_kernel) and
// solution/cross_entropy.py:48-90 (fused_ce_kernel). Per row z[0..V):
//   m = max z, s = sum exp(z - m), t = sum exp(z - m) * z
//   lse = m + log s ; entropy = lse - t / s ; argmax = first index of the maximum
//   loss = labelled ? lse - z[target] : 0
//   dz   = (exp(z - lse) - [v == target]) * (labelled ? grad_scale : 0)   (in place)
//
// HBM-bound: sweep 1 reads the row, sweep 2 reads it again and overwrites it with dz.
// One 512-thread workgroup per row; each thread walks 8-element (16 B) chunks with a stride
// of the workgroup, keeping a running (m, s, t, best, best_idx) per thread, rescaling once
// per chunk. Threads combine through wave butterflies and one LDS exchange.
//
// Second reads stay on chip: each thread keeps its first chunks of the row (the row's first
// 64 KiB) in LDS for sweep 2, and the 64 KiB per workgroup hold the GPU at two rows per CU,
// so the 512 rows in flight (156 MB at the Qwen2 vocabulary, 151936 x 2 B a row) stay inside
// the 256 MB MALL and the rest of sweep 2 reads from there (1.15 ms for 8192 x 151936 bf16, against
// 1.45 ms with four rows per CU: the 1024 rows in flight spilled the MALL). Both sweeps load 4
// chunks, then do their arithmetic as one piece: one maximum, one rescaling, one test for small
// exponents, the target's entry by itself. With a maximum and its index, a scaled exponential
// and a 64-bit target test per element the vector ALU took as long as the memory (4096 x 151936
// bf16 641 us, 512 x 151936 82.6, 1000 x 32000 47.4; now 594, 69, 35). 8 chunks at a time need
// more than the 128 registers of four waves per SIMD: 690, 77, 47. Rows that go element by element
// (V or a row's address not a multiple of 8 elements) take 4 elements as such a piece: 4096 x 50257
// bf16 253 us; one at a time 482, against 426 with the per-element arithmetic above.
#include <type_traits>

#include "ql_vec.h"

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr float kLog2e = 1.4426950408889634f;

struct RowStat {
  float m, s, t, best;
  int64_t best_idx;
};

QL_DEV void merge(RowStat& a, const RowStat& b) {
  // (m, s, t): rescale both sides to the larger max. best: larger value, then lower index.
  const float m = fmaxf(a.m, b.m);
  const float fa = (a.m == -INFINITY) ? 0.f : exp2f((a.m - m) * kLog2e);
  const float fb = (b.m == -INFINITY) ? 0.f : exp2f((b.m - m) * kLog2e);
  a.s = a.s * fa + b.s * fb;
  a.t = a.t * fa + b.t * fb;
  a.m = m;
  if (b.best > a.best || (b.best == a.best && b.best_idx < a.best_idx)) {
    a.best = b.best;
    a.best_idx = b.best_idx;
  }
}

QL_DEV RowStat shfl_stat(const RowStat& v, int off) {
  RowStat r;
  r.m = __shfl_xor(v.m, off, 64);
  r.s = __shfl_xor(v.s, off, 64);
  r.t = __shfl_xor(v.t, off, 64);
  r.best = __shfl_xor(v.best, off, 64);
  r.best_idx = __shfl_xor(v.best_idx, off, 64);
  return r;
}

// v[j] = exp2f(v[j]). exp2f is v_exp_f32 except below -126, where it scales the argument up and
// the (subnormal) result down, five more instructions per element. A wave without such an
// element takes v_exp_f32 alone, with the same bits.
template <int N>
QL_DEV void exp2_chunk(float* v) {
  float lo = v[0];
#pragma unroll
  for (int j = 1; j < N; ++j) lo = fminf(lo, v[j]);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(lo < -126.f) == 0, 1)) {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = __builtin_amdgcn_exp2f(v[j]);
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = exp2f(v[j]);
  }
}

constexpr int kCacheBytes = 64 * 1024;  // LDS row cache per workgroup (dynamic)
constexpr int kUnroll = 4;  // chunk loads in flight per thread

// VW = 8: 8-element chunks (V % 8 == 0, 16-B aligned rows), 16-bit ones cached in LDS;
// VW = 1: one element per step, no cache.
template <int DT, int VW>
__global__ __launch_bounds__(kThreads) void ce_rows_kernel(
    typename Elem<DT>::T* __restrict__ logits, int64_t row_stride, int64_t V,
    const int64_t* __restrict__ target, float* __restrict__ loss, float* __restrict__ entropy,
    int32_t* __restrict__ correct, int64_t* __restrict__ pred, int ignore_mode, int write_grad,
    float grad_scale, const float* __restrict__ grad_scale_dev) {
  extern __shared__ uint4 cache[];  // kCacheBytes when VW == 8
  __shared__ RowStat part[kWaves];
  __shared__ float lse_sh;
  constexpr bool kCached = VW == 8 && DT != QL_F32;  // a 16-B chunk per 8 elements
  constexpr int64_t kCacheChunks = kCached ? kCacheBytes / 16 : 0;
  constexpr int U = kUnroll;
  const int64_t row = blockIdx.x;
  auto* z = logits + row * row_stride;
  const int64_t tgt = target[row];
  const bool labelled = ignore_mode == 0 ? (tgt >= 0) : (tgt != -100);
  const int64_t nchunk = V / VW;
  auto load = [&](int64_t c, float* v) {  // sweep 2
    if constexpr (kCached) {
      const uint4 raw = c < kCacheChunks ? cache[c] : *reinterpret_cast<const uint4*>(z + 8 * c);
      Vec8<DT>::unpack(raw, v);
    } else if constexpr (VW == 8) {
      Vec8<DT>::load(z + 8 * c, v);
    } else {
      v[0] = Elem<DT>::to_f32(z[c]);
    }
  };
  auto load_keep = [&](int64_t c, float* v) {  // sweep 1: also fills the cache
    if constexpr (kCached) {
      const uint4 raw = *reinterpret_cast<const uint4*>(z + 8 * c);
      if (c < kCacheChunks) cache[c] = raw;
      Vec8<DT>::unpack(raw, v);
    } else {
      load(c, v);
    }
  };

  RowStat st{-INFINITY, 0.f, 0.f, -INFINITY, 0};
  int64_t best_c = -1;  // the first chunk with this thread's maximum
  // N chunks, c and every kThreads-th after it: one rescaling of the sums for all of them
  auto absorb = [&](auto count, const float (*v)[VW], int64_t c) {
    constexpr int N = decltype(count)::value;
    float cm[N], gm = -INFINITY;
#pragma unroll
    for (int u = 0; u < N; ++u) {
      cm[u] = v[u][0];
#pragma unroll
      for (int j = 1; j < VW; ++j) cm[u] = fmaxf(cm[u], v[u][j]);
      cm[u] = v[u][0] == v[u][0] ? cm[u] : v[u][0];  // one that starts with NaN is never the maximum
      gm = fmaxf(gm, cm[u]);
    }
    if (gm > st.best) {
      st.best = gm;
#pragma unroll
      for (int u = N - 1; u >= 0; --u) best_c = cm[u] == gm ? c + u * kThreads : best_c;
    }
    const float m = fmaxf(st.m, gm);
    const float alpha = (st.m == -INFINITY) ? 0.f : exp2f((st.m - m) * kLog2e);
    float e[N * VW], es = 0.f, et = 0.f;
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int j = 0; j < VW; ++j) e[u * VW + j] = (v[u][j] - m) * kLog2e;
    exp2_chunk<N * VW>(e);
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int j = 0; j < VW; ++j) {
        es += e[u * VW + j];
        et += e[u * VW + j] * v[u][j];
      }
    st.s = st.s * alpha + es;
    st.t = st.t * alpha + et;
    st.m = m;
  };
  // Sweep 1, in increasing chunk order per thread (the first maximum wins): U loads, then
  // their arithmetic; chunks below kCacheChunks are also kept in LDS for sweep 2.
  int64_t c0 = threadIdx.x;
  for (; c0 + (U - 1) * kThreads < nchunk; c0 += U * kThreads) {
    float v[U][VW];
#pragma unroll
    for (int u = 0; u < U; ++u) load_keep(c0 + u * kThreads, v[u]);
    absorb(std::integral_constant<int, U>{}, v, c0);
  }
  for (int64_t c = c0; c < nchunk; c += kThreads) {
    float v[1][VW];
    load_keep(c, v[0]);
    absorb(std::integral_constant<int, 1>{}, v, c);
  }
  if (best_c >= 0) {  // the first element of that chunk that holds it
    float v[VW];
    load(best_c, v);
    int j = VW - 1;
#pragma unroll
    for (int i = VW - 2; i >= 0; --i) j = v[i] == st.best ? i : j;
    st.best_idx = best_c * VW + j;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) merge(st, shfl_stat(st, off));
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) part[wid] = st;
  __syncthreads();
  if (threadIdx.x == 0) {
    RowStat a = part[0];
    for (int i = 1; i < kWaves; ++i) merge(a, part[i]);
    const float lse = a.m + logf(a.s);
    lse_sh = lse;
    // A label outside [0, V) is never read (the loss becomes NaN instead of a stray load).
    const bool in_range = tgt >= 0 && tgt < V;
    const float zt = (labelled && in_range) ? Elem<DT>::to_f32(z[tgt]) : NAN;
    loss[row] = labelled ? lse - zt : 0.f;
    entropy[row] = lse - a.t / a.s;
    if (correct) correct[row] = (labelled && a.best_idx == tgt) ? 1 : 0;
    if (pred) pred[row] = a.best_idx;
  }
  if (!write_grad) return;
  __syncthreads();
  const float lse = lse_sh;
  const float gs = labelled ? (grad_scale_dev ? *grad_scale_dev : grad_scale) : 0.f;
  auto emit = [&](auto count, float (*v)[VW], int64_t c) {
    constexpr int N = decltype(count)::value;
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int j = 0; j < VW; ++j) v[u][j] = (v[u][j] - lse) * kLog2e;
    exp2_chunk<N * VW>(v[0]);
#pragma unroll
    for (int u = 0; u < N; ++u, c += kThreads) {
      const int64_t hot = tgt - c * VW;
      if (hot >= 0 && hot < VW) {  // one thread of the row, once
#pragma unroll
        for (int j = 0; j < VW; ++j) v[u][j] = j == (int)hot ? v[u][j] - 1.f : v[u][j];
      }
#pragma unroll
      for (int j = 0; j < VW; ++j) v[u][j] *= gs;
      if constexpr (VW == 8) Vec8<DT>::store(z + 8 * c, v[u]);
      else z[c] = Elem<DT>::from_f32(v[u][0]);
    }
  };
  // Sweep 2: every thread rewrites the chunks it read (its cached ones from LDS), U loads
  // ahead of their arithmetic.
  c0 = threadIdx.x;
  for (; c0 + (U - 1) * kThreads < nchunk; c0 += U * kThreads) {
    float v[U][VW];
#pragma unroll
    for (int u = 0; u < U; ++u) load(c0 + u * kThreads, v[u]);
    emit(std::integral_constant<int, U>{}, v, c0);
  }
  for (int64_t c = c0; c < nchunk; c += kThreads) {
    float v[1][VW];
    load(c, v[0]);
    emit(std::integral_constant<int, 1>{}, v, c);
  }
}

template <int DT>
int launch_ce(void* logits, int64_t rs, int64_t n_rows, int64_t V, const int64_t* target,
              float* loss, float* entropy, int32_t* correct, int64_t* pred, int ignore_mode,
              int write_grad, float grad_scale, const float* grad_scale_dev, hipStream_t s) {
  using T = typename Elem<DT>::T;
  const bool vec = (V % 8) == 0 && ql_aligned(logits, 16) && ((rs * ql_elem_size(DT)) % 16) == 0;
  if (vec)
    hipLaunchKernelGGL((ce_rows_kernel<DT, 8>), dim3((unsigned)n_rows), dim3(kThreads),
                       DT == QL_F32 ? 0 : kCacheBytes, s,
                       (T*)logits, rs, V, target, loss, entropy, correct, pred, ignore_mode,
                       write_grad, grad_scale, grad_scale_dev);
  else
    hipLaunchKernelGGL((ce_rows_kernel<DT, 1>), dim3((unsigned)n_rows), dim3(kThreads), 0, s,
                       (T*)logits, rs, V, target, loss, entropy, correct, pred, ignore_mode,
                       write_grad, grad_scale, grad_scale_dev);
  return ql_launch_status();
}

int ce_rows(void* logits, int logits_dtype, int64_t row_stride, int64_t n_rows, int64_t vocab,
            const int64_t* target, float* loss, float* entropy, int32_t* correct, int64_t* pred,
            int ignore_mode, int write_grad, float grad_scale, const float* grad_scale_dev,
            ql_stream_t stream) {
  if (n_rows < 0 || vocab <= 0 || n_rows > UINT32_MAX) return QL_EINVAL;
  if (ignore_mode != 0 && ignore_mode != 1) return QL_EINVAL;
  if (!ql_valid_dtype(logits_dtype)) return QL_EDTYPE;
  if (n_rows == 0) return QL_OK;
  if (!logits || !target || !loss || !entropy) return QL_EINVAL;
  QL_DISPATCH_DTYPE(logits_dtype, DT,
                    return launch_ce<DT>(logits, row_stride, n_rows, vocab, target, loss, entropy,
                                         correct, pred, ignore_mode, write_grad, grad_scale,
                                         grad_scale_dev, static_cast<hipStream_t>(stream)));
  return QL_EDTYPE;
}

}  // namespace

extern "C" int qlora_ce_rows(void* logits, int logits_dtype, int64_t row_stride, int64_t n_rows,
                             int64_t vocab, const int64_t* target, float* loss, float* entropy,
                             int32_t* correct, int64_t* pred, int ignore_mode, int write_grad,
                             float grad_scale, ql_stream_t stream) {
  return ce_rows(logits, logits_dtype, row_stride, n_rows, vocab, target, loss, entropy, correct,
                 pred, ignore_mode, write_grad, grad_scale, nullptr, stream);
}

extern "C" int qlora_ce_rows_scale_ptr(void* logits, int logits_dtype, int64_t row_stride,
                                       int64_t n_rows, int64_t vocab, const int64_t* target,
                                       float* loss, float* entropy, int32_t* correct,
                                       int64_t* pred, int ignore_mode, int write_grad,
                                       const float* grad_scale, ql_stream_t stream) {
  if (write_grad && !grad_scale) return QL_EINVAL;
  return ce_rows(logits, logits_dtype, row_stride, n_rows, vocab, target, loss, entropy, correct,
                 pred, ignore_mode, write_grad, 0.f, write_grad ? grad_scale : nullptr, stream);
}
