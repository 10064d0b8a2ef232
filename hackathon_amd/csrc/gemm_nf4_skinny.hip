// The 4-bit linear for a few rows of x (decoding, small evaluation batches), for gfx950:
//
//   C[m, n] = alpha * (sum_k x[m, k] * W[n, k] + sum_j a2[m, j] * b2[n, j]) (+ bias[n])
//
// W [N, K] is the packed NF4 weight, rounded to the 16-bit compute dtype weight by weight as
// qlora_nf4_dequant writes it (scale = code2[q] * absmax2, then + offset; product rounded to
// fp32, then to 16 bits). This is F.linear on the dequantised weight (solution/nf4.py:95-102)
// with the rank-16 adapter term (solution/lora.py:49-60,172) as a second K segment.
//
// What bounds it. With M <= kSkinnyMaxRows rows the products are nothing and W's 0.52 bytes a
// weight have to arrive once: 35 MB at 18944 x 3584, 7 us at 5 TB/s. Turning nibbles into MFMA
// operands costs about five vector operations a weight, 10 us of the whole chip for that
// weight: the vector units, not HBM, are the bound. The 256 x 256 tiles of the large GEMM reach
// neither: at 4 rows each of their 74 workgroups (on 256 CUs) dequantises 256 rows through LDS
// between barriers, for rows of x that are 98% padding, and splits K through memory.
// Measured per call (HIP graph, 3 rotated weights, the 64-column segment included), large tile
// -> this kernel: 18944 x 3584 50.6 -> 17.5 us at 4 rows, 52.5 -> 30.0 at 32; 3584 x 18944
// 48.5 -> 17.0 and 51.5 -> 43.8; 3584 x 3584 27.5 -> 6.6 and 30.2 -> 12.3; 4864 x 896
// 37.0 -> 4.4 and 37.8 -> 7.2. Past 32 rows the loads of x catch up with the large tile.
//
// Split. A workgroup owns 16 R rows of W and the whole K; its waves take the 256-k chunks in
// turn and meet once, in LDS, at the end. No partial results go to memory and no second launch
// sums them. A lane holds 64 consecutive weights of one row (32 B, one absmax block), so the
// block's 16 products are made once per 64 weights and every weight is then a byte-permute
// lookup, and the four lanes of a row read one whole 128-B line. The eight 8-weight words are
// MFMA operands as they lie: v_mfma_f32_16x16x32 wants 8 consecutive k per lane, and the sum
// over k does not care which lane holds which. The lookups give the even weights of a word and
// then the odd ones; x is permuted alike (once per R row groups) instead of un-permuting W.
// A whole LoRA layer without gradients (qlora_nf4_lora_few) is this kernel and one small
// down-projection before it, both reading the adapter's fp32 factors: the packed copies, the
// reduce of the down-projection and the zero-padded u are for the training path. At 4 rows of
// 18944 x 3584: 4 launches and 34 us of kernels -> 2 and 22 us; the layer's call 80.7 -> 35.5 us.
// R = 2 (32 rows) halves the loads of x per weight and is taken when that still gives every CU
// a workgroup; the waves per workgroup grow with K so that a wave has about four chunks.
#include "gemm_nt.h"
#include "ql_common.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

constexpr int kChunk = 256;     // k per wave step: 64 per lane of a row's four lanes

template <int DT> QL_DEV f32x4_t mfma(const uint4& a, const uint4& b, f32x4_t c);
template <> QL_DEV f32x4_t mfma<QL_BF16>(const uint4& a, const uint4& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                  __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <> QL_DEV f32x4_t mfma<QL_F16>(const uint4& a, const uint4& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                 __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// The product must reach fp32 before the 16-bit conversion (the backend would otherwise fuse
// multiply and conversion into one rounding).
QL_DEV float rounded32(float x) {
  asm("" : "+v"(x));
  return x;
}

template <int IT> QL_DEV uint32_t pack2(float lo, float hi) {
  if constexpr (IT == QL_BF16) return pack_bf16x2(lo, hi);
  else return pack_f16x2(lo, hi);
}

// The 16 products nf4[c] * s of a block in the compute dtype, as planes of their low and high
// bytes (four entries a word).
struct Planes {
  uint32_t lo[4], hi[4];
};

template <int IT> QL_DEV Planes make_planes(const float (&nf4)[16], float s) {
#pragma clang fp contract(off)
  uint32_t pair[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    pair[i] = pack2<IT>(rounded32(nf4[2 * i] * s), rounded32(nf4[2 * i + 1] * s));
  Planes p;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    p.lo[j] = __builtin_amdgcn_perm(pair[2 * j + 1], pair[2 * j], 0x06040200u);
    p.hi[j] = __builtin_amdgcn_perm(pair[2 * j + 1], pair[2 * j], 0x07050301u);
  }
  return p;
}

// Byte j: entry sel.byte[j] of a plane; sel7 the low three bits of each index, pick byte j = j,
// or j + 4 where the index is 8 or more.
QL_DEV uint32_t lookup(const uint32_t (&plane)[4], uint32_t sel7, uint32_t pick) {
  const uint32_t a = __builtin_amdgcn_perm(plane[1], plane[0], sel7);
  const uint32_t b = __builtin_amdgcn_perm(plane[3], plane[2], sel7);
  return __builtin_amdgcn_perm(b, a, pick);
}

// The 8 weights of packed word d (byte i: weight 2i in the high nibble, 2i + 1 in the low one)
// in the order 0 2 4 6 1 3 5 7. `ident` is 0x03020100 in a register: with it and the mask the
// insertion of the index's top bit is one v_bfi_b32 (with two literals it would be two).
QL_DEV uint4 weights_of(const Planes& p, uint32_t d, uint32_t ident) {
  const uint32_t sel_e = (d >> 4) & 0x07070707u, sel_o = d & 0x07070707u;
  const uint32_t pick_e = ((d >> 5) & 0x04040404u) | (ident & ~0x04040404u);
  const uint32_t pick_o = ((d >> 1) & 0x04040404u) | (ident & ~0x04040404u);
  const uint32_t le = lookup(p.lo, sel_e, pick_e), he = lookup(p.hi, sel_e, pick_e);
  const uint32_t lo = lookup(p.lo, sel_o, pick_o), ho = lookup(p.hi, sel_o, pick_o);
  return make_uint4(__builtin_amdgcn_perm(he, le, 0x05010400u),
                    __builtin_amdgcn_perm(he, le, 0x07030602u),
                    __builtin_amdgcn_perm(ho, lo, 0x05010400u),
                    __builtin_amdgcn_perm(ho, lo, 0x07030602u));
}

// 8 consecutive 16-bit values in that order.
QL_DEV uint4 even_odd(const uint4& v) {
  return make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u),
                    __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
                    __builtin_amdgcn_perm(v.y, v.x, 0x07060302u),
                    __builtin_amdgcn_perm(v.w, v.z, 0x07060302u));
}

struct SkinnyArgs {
  const uint16_t* x;
  int64_t ldx;
  const uint8_t* packed;
  const void* absmax;    // uint8 codes (nested) or fp32
  const float* code2;
  const float* absmax2;
  const float* nf4;
  float offset;
  int log2_bs, log2_bs2;
  const uint16_t *a2, *b2;
  int64_t lda2, ldb2;
  int k2;                // 0 or 64
  // instead of a2 / b2: x's down-projections as fp32 partials [u_splits][M][16], and the
  // adapter's B [N, 16] in fp32, scaled here
  const float *u_part, *lora_b;
  int u_splits;
  float scaling;
  uint16_t* c;
  int64_t ldc;
  const uint16_t* bias;
  int64_t M, N, K;
  float alpha;
};

// One lane's weights of a chunk: 64 of each of R rows, and their absmax.
template <int R> struct Stage {
  uint4 w[R][2];
  uint32_t code[R];
  float scale2[R];
};

template <bool NESTED, int R>
QL_DEV void load_weights(Stage<R>& st, const SkinnyArgs& p, const int64_t (&wrow)[R], int64_t k) {
  const int64_t kk = k < p.K ? k : 0;   // K % 64 == 0: a lane's 64 k are all in or all out
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t w0 = wrow[r] + kk;
    const uint4* q = reinterpret_cast<const uint4*>(p.packed + (w0 >> 1));
    st.w[r][0] = q[0];
    st.w[r][1] = q[1];
    const int64_t blk = w0 >> p.log2_bs;
    if constexpr (NESTED) {
      st.code[r] = static_cast<const uint8_t*>(p.absmax)[blk];
      st.scale2[r] = p.absmax2[blk >> p.log2_bs2];
    } else {
      st.code[r] = __float_as_uint(static_cast<const float*>(p.absmax)[blk]);
      st.scale2[r] = 0.f;
    }
  }
}

// 64 values of MT rows of x into the lanes of rows below M; the others keep the zeros they were
// given before the loop. Past K (in the last chunk only) a lane gets zeros too.
template <int MT>
QL_DEV void load_x(uint4 (&x)[MT][8], const uint16_t* const (&xrow)[MT], const bool (&xok)[MT],
                   int64_t k, int64_t K) {
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (xok[i]) {
      if (k < K) {
#pragma unroll
        for (int t = 0; t < 8; ++t)
          x[i][t] = *reinterpret_cast<const uint4*>(xrow[i] + k + 8 * t);
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) x[i][t] = make_uint4(0u, 0u, 0u, 0u);
      }
    }
  }
}

// Waves a workgroup may have: 16 need 128 registers or fewer a lane, which two 16-row groups of
// x (64 registers) do not leave.
template <int MT> constexpr int max_waves() { return MT == 1 ? 16 : 8; }

template <int IT, bool NESTED, int R, int MT>
__global__ __launch_bounds__(64 * max_waves<MT>()) void gemm_nf4_skinny_kernel(SkinnyArgs p) {
#pragma clang fp contract(off)
  __shared__ float code2_lds[NESTED ? 256 : 1];
  __shared__ f32x4_t red[max_waves<MT>() * R * MT * 64];
  const int lane = threadIdx.x & 63, row = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  const int64_t n0 = (int64_t)blockIdx.x * 16 * R;

  int64_t wrow[R];  // weight index of (row, 0); rows past N read the last one and are not stored
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t n = n0 + 16 * r + row;
    wrow[r] = (n < p.N ? n : p.N - 1) * p.K;
  }
  const uint16_t* xrow[MT];
  bool xok[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int64_t m = 16 * i + row;
    xok[i] = m < p.M;
    xrow[i] = p.x + (xok[i] ? m : 0) * p.ldx;
  }
  float nf4[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) nf4[i] = p.nf4[i];

  const int64_t chunks = (p.K + kChunk - 1) / kChunk;
  Stage<R> st;
  if (wave < chunks) load_weights<NESTED, R>(st, p, wrow, (int64_t)wave * kChunk + 64 * quad);
  if constexpr (NESTED) {
    for (int t = threadIdx.x; t < 256; t += blockDim.x) code2_lds[t] = p.code2[t];
    __syncthreads();
  }

  f32x4_t acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[r][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  uint32_t ident = 0x03020100u;
  asm("" : "+v"(ident));
  uint4 x[MT][8];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < 8; ++t) x[i][t] = make_uint4(0u, 0u, 0u, 0u);
  for (int64_t c = wave; c < chunks; c += waves) {
    // x of this chunk (from the caches) goes out before the next chunk's weights (from HBM):
    // loads complete in issue order, so waiting for x leaves the weights in flight
    const Stage<R> now = st;
    load_x<MT>(x, xrow, xok, c * kChunk + 64 * quad, p.K);
    if (c + waves < chunks)
      load_weights<NESTED, R>(st, p, wrow, (c + waves) * kChunk + 64 * quad);
    const bool in = c * kChunk + 64 * quad < p.K;
    Planes pl[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float s;
      if constexpr (NESTED) {
        s = code2_lds[now.code[r]] * now.scale2[r];  // two fp32 roundings
        s = s + p.offset;
      } else {
        s = __uint_as_float(now.code[r]);
      }
      pl[r] = make_planes<IT>(nf4, in ? s : 0.f);  // past K: zeros against zeros
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      uint4 xv[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) xv[i] = even_odd(x[i][t]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint4& h = now.w[r][t >> 2];
        const uint32_t d = (t & 3) == 0 ? h.x : (t & 3) == 1 ? h.y : (t & 3) == 2 ? h.z : h.w;
        const uint4 wv = weights_of(pl[r], d, ident);
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[r][i] = mfma<IT>(wv, xv[i], acc[r][i]);
      }
    }
  }
  // the rank-16 segment (64 columns, zero-padded): two 32-k products of the last wave, which has
  // the fewest chunks
  if (p.k2 && wave == waves - 1) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      uint4 av[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        av[i] = make_uint4(0u, 0u, 0u, 0u);
        if (xok[i])
          av[i] = *reinterpret_cast<const uint4*>(p.a2 + (16 * i + row) * p.lda2 + 32 * t +
                                                  8 * quad);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int64_t n = n0 + 16 * r + row;
        const uint4 bv = *reinterpret_cast<const uint4*>(
            p.b2 + (n < p.N ? n : p.N - 1) * p.ldb2 + 32 * t + 8 * quad);
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[r][i] = mfma<IT>(bv, av[i], acc[r][i]);
      }
    }
  }
  // or the adapter in fp32: u = the partials in split order, rounded to the compute dtype, against
  // s B rounded likewise (16 of a product's 32 k: the upper lanes hold zeros)
  if (p.u_part && wave == waves - 1) {
    const bool half = quad < 2;
    uint4 uv[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (half && xok[i]) {
        const float* q = p.u_part + (int64_t)(16 * i + row) * 16 + 8 * quad;
        for (int z = 0; z < p.u_splits; ++z, q += p.M * 16) {
          const float4 lo = reinterpret_cast<const float4*>(q)[0];
          const float4 hi = reinterpret_cast<const float4*>(q)[1];
          const float w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += w[e];
        }
      }
      uv[i] = make_uint4(pack2<IT>(v[0], v[1]), pack2<IT>(v[2], v[3]), pack2<IT>(v[4], v[5]),
                         pack2<IT>(v[6], v[7]));
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t n = n0 + 16 * r + row;
      uint4 bv = make_uint4(0u, 0u, 0u, 0u);
      if (half) {
        const float4* q = reinterpret_cast<const float4*>(p.lora_b + (n < p.N ? n : p.N - 1) * 16 +
                                                          8 * quad);
        const float4 lo = q[0], hi = q[1];
        const float s = p.scaling;
        bv = make_uint4(pack2<IT>(rounded32(lo.x * s), rounded32(lo.y * s)),
                        pack2<IT>(rounded32(lo.z * s), rounded32(lo.w * s)),
                        pack2<IT>(rounded32(hi.x * s), rounded32(hi.y * s)),
                        pack2<IT>(rounded32(hi.z * s), rounded32(hi.w * s)));
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[r][i] = mfma<IT>(bv, uv[i], acc[r][i]);
    }
  }
  // sum the waves in wave order; lane l of block (r, i) holds x row 16 i + l % 16, columns
  // n0 + 16 r + 4 (l / 16) .. + 3
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int i = 0; i < MT; ++i) red[(wave * R * MT + r * MT + i) * 64 + lane] = acc[r][i];
  __syncthreads();
  for (int e = threadIdx.x; e < R * MT * 64; e += blockDim.x) {
    f32x4_t s = red[e];
    for (int w = 1; w < waves; ++w) {
      const f32x4_t v = red[w * R * MT * 64 + e];
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += v[j];
    }
    const int l = e & 63, blk = e >> 6;
    const int64_t m = 16 * (blk % MT) + (l & 15);
    const int64_t n = n0 + 16 * (blk / MT) + 4 * (l >> 4);
    if (m >= p.M || n >= p.N) continue;
    uint16_t* cp = p.c + m * p.ldc + n;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = p.alpha * s[j];
      if (p.bias && n + j < p.N) v[j] += Elem<IT>::to_f32(p.bias[n + j]);
    }
    if (n + 4 <= p.N && ((uintptr_t)cp & 7) == 0) {
      *reinterpret_cast<uint2*>(cp) = make_uint2(pack2<IT>(v[0], v[1]), pack2<IT>(v[2], v[3]));
    } else {
      for (int j = 0; j < 4 && n + j < p.N; ++j) cp[j] = Elem<IT>::from_f32(v[j]);
    }
  }
}

template <int IT, bool NESTED, int R, int MT>
int launch(const SkinnyArgs& p, int waves, hipStream_t s) {
  hipLaunchKernelGGL((gemm_nf4_skinny_kernel<IT, NESTED, R, MT>),
                     dim3((unsigned)((p.N + 16 * R - 1) / (16 * R))), dim3(64 * waves), 0, s, p);
  return ql_launch_status();
}

template <int IT, bool NESTED>
int launch_rows(const SkinnyArgs& p, hipStream_t s) {
  const int64_t chunks = (p.K + kChunk - 1) / kChunk;
  const int most = p.M <= 16 ? max_waves<1>() : max_waves<2>();
  int waves = 4;
  while (waves < most && chunks > 4 * waves) waves *= 2;
  // two 16-row groups per load of x: where x has enough rows for its loads to count and
  // 32-row workgroups still reach every CU (18944 x 3584: 16.1 against 17.6 us at 1 row for
  // one group, 24.3 against 20.8 at 16 rows, 41.5 against 30.1 at 32)
  const bool wide = p.M > 8 && p.N >= 32 * 256;
  if (p.M <= 16) return wide ? launch<IT, NESTED, 2, 1>(p, waves, s) : launch<IT, NESTED, 1, 1>(p, waves, s);
  return wide ? launch<IT, NESTED, 2, 2>(p, waves, s) : launch<IT, NESTED, 1, 2>(p, waves, s);
}

// u_part[split][m][r] = sum over the split's k of x[m, k] A[r, k], A [16, K] in fp32 rounded to the
// compute dtype on the way (the values a packed copy of A would hold, without the launch and the
// copy). One workgroup per split; its four waves take 32-k steps in turn, up to four of them in
// flight, and meet in LDS.
constexpr int kDownWaves = 4, kDownUnroll = 4;

template <int IT, int MT>
__global__ __launch_bounds__(64 * kDownWaves) void lora_down_few_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const float* __restrict__ A, int64_t M, int64_t K,
    int64_t k_per_split, float* __restrict__ u_part) {
  __shared__ f32x4_t red[kDownWaves * MT * 64];
  const int lane = threadIdx.x & 63, row = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t kb = (int64_t)blockIdx.x * k_per_split;
  const int64_t ke = kb + k_per_split < K ? kb + k_per_split : K;
  f32x4_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int64_t k0 = kb + 32 * wave; k0 < ke; k0 += 32 * kDownWaves * kDownUnroll) {
    float4 a[kDownUnroll][2];
    uint4 xv[kDownUnroll][MT];
#pragma unroll
    for (int u = 0; u < kDownUnroll; ++u) {  // K and the splits are multiples of 32
      const int64_t k = k0 + 32 * kDownWaves * u;
      const bool in = k < ke;
      const int64_t kk = (in ? k : kb) + 8 * quad;
      const float4* q = reinterpret_cast<const float4*>(A + row * K + kk);
      a[u][0] = q[0];
      a[u][1] = q[1];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        xv[u][i] = make_uint4(0u, 0u, 0u, 0u);
        if (in && 16 * i + row < M)
          xv[u][i] = *reinterpret_cast<const uint4*>(x + (16 * i + row) * ldx + kk);
      }
      if (!in) a[u][0] = a[u][1] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < kDownUnroll; ++u) {
      const uint4 av = make_uint4(pack2<IT>(a[u][0].x, a[u][0].y), pack2<IT>(a[u][0].z, a[u][0].w),
                                  pack2<IT>(a[u][1].x, a[u][1].y), pack2<IT>(a[u][1].z, a[u][1].w));
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] = mfma<IT>(av, xv[u][i], acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) red[(wave * MT + i) * 64 + lane] = acc[i];
  __syncthreads();
  // lane l of block i: x row 16 i + l % 16, adapter rows 4 (l / 16) .. + 3
  for (int e = threadIdx.x; e < MT * 64; e += 64 * kDownWaves) {
    f32x4_t s = red[e];
#pragma unroll
    for (int w = 1; w < kDownWaves; ++w)
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += red[w * MT * 64 + e][j];
    const int64_t m = 16 * (e >> 6) + (e & 15);
    if (m < M)
      *reinterpret_cast<float4*>(u_part + ((int64_t)blockIdx.x * M + m) * 16 + 4 * ((e & 63) >> 4)) =
          make_float4(s[0], s[1], s[2], s[3]);
  }
}

// Splits of the down-projection: a wave's four steps in flight cover 512 k a workgroup; at most
// eight, so that the few kilobytes of partials stay a detail of every workgroup that sums them.
int64_t down_k_per_split(int64_t K) {
  int64_t splits = (K + 511) / 512;
  if (splits > 8) splits = 8;
  return ((K / 32 + splits - 1) / splits) * 32;
}

template <int IT>
int launch_down(const void* x, int64_t ldx, const float* A, int64_t M, int64_t K, float* u_part,
                hipStream_t s) {
  const int64_t kps = down_k_per_split(K);
  const dim3 grid((unsigned)((K + kps - 1) / kps)), block(64 * kDownWaves);
  if (M <= 16)
    hipLaunchKernelGGL((lora_down_few_kernel<IT, 1>), grid, block, 0, s, (const uint16_t*)x, ldx, A,
                       M, K, kps, u_part);
  else
    hipLaunchKernelGGL((lora_down_few_kernel<IT, 2>), grid, block, 0, s, (const uint16_t*)x, ldx, A,
                       M, K, kps, u_part);
  return ql_launch_status();
}

}  // namespace

int ql_gemm_nf4_skinny(int64_t M, int64_t N, int64_t K, const void* A, int64_t lda,
                       const uint8_t* packed, const void* absmax, int nested, const float* code2,
                       const float* absmax2, float offset, int log2_bs, int log2_bs2,
                       const float* nf4_table, int64_t K2, const void* A2, int64_t lda2,
                       const void* B2, int64_t ldb2, int in_dtype, void* C, int64_t ldc,
                       const void* bias, float alpha, hipStream_t s) {
  if (M > kSkinnyMaxRows || (K2 != 0 && K2 != 64)) return QL_ESHAPE;
  const SkinnyArgs p{(const uint16_t*)A, lda, packed, absmax, code2, absmax2, nf4_table, offset,
                     log2_bs, log2_bs2, (const uint16_t*)A2, (const uint16_t*)B2, lda2, ldb2,
                     (int)K2, nullptr, nullptr, 0, 0.f, (uint16_t*)C, ldc, (const uint16_t*)bias, M, N, K, alpha};
  if (in_dtype == QL_BF16)
    return nested ? launch_rows<QL_BF16, true>(p, s) : launch_rows<QL_BF16, false>(p, s);
  return nested ? launch_rows<QL_F16, true>(p, s) : launch_rows<QL_F16, false>(p, s);
}

extern "C" int64_t qlora_nf4_lora_few_workspace_size(int64_t M, int64_t K) {
  if (M <= 0 || M > kSkinnyMaxRows || K <= 0 || K % 64) return 0;
  const int64_t kps = down_k_per_split(K);
  return (K + kps - 1) / kps * M * 16 * (int64_t)sizeof(float);
}

extern "C" int qlora_nf4_lora_few(int64_t M, int64_t N, int64_t K, const void* x, int64_t ldx,
                                  const uint8_t* packed, const void* absmax, int nested,
                                  const float* code2, const float* absmax2, float offset,
                                  int blocksize, int blocksize2, const float* nf4_table,
                                  const float* lora_a, const float* lora_b, float scaling,
                                  int dtype, void* C, int64_t ldc, const void* bias,
                                  void* workspace, int64_t workspace_bytes, ql_stream_t stream) {
  if (M < 0 || N < 0 || K < 0 || workspace_bytes < 0) return QL_EINVAL;
  if (dtype != QL_BF16 && dtype != QL_F16) return QL_EDTYPE;
  if (M == 0 || N == 0) return QL_OK;
  if (!x || !packed || !absmax || !nf4_table || !lora_a || !lora_b || !C) return QL_EINVAL;
  if (nested && (!code2 || !absmax2)) return QL_EINVAL;
  if (M > kSkinnyMaxRows || K <= 0 || K % 64) return QL_ESHAPE;
  const auto log2_exact = [](int64_t v) {
    int l = 0;
    while ((int64_t(1) << l) < v) ++l;
    return v > 0 && (int64_t(1) << l) == v ? l : -1;
  };
  const int log2_bs = log2_exact(blocksize), log2_bs2 = nested ? log2_exact(blocksize2) : 0;
  if (log2_bs < 6 || K % blocksize || log2_bs2 < 0) return QL_EINVAL;
  if (ldx < K || ldc < N || N > (int64_t(1) << 30)) return QL_ESHAPE;
  if (ldx % 8 || !ql_aligned(x, 16) || !ql_aligned(packed, 16) || !ql_aligned(C, 2) ||
      !ql_aligned(lora_a, 16) || !ql_aligned(lora_b, 16) || (bias && !ql_aligned(bias, 2)))
    return QL_EALIGN;
  if (!workspace || !ql_aligned(workspace, 16) ||
      workspace_bytes < qlora_nf4_lora_few_workspace_size(M, K))
    return QL_EINVAL;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  float* part = static_cast<float*>(workspace);
  const int st = dtype == QL_BF16 ? launch_down<QL_BF16>(x, ldx, lora_a, M, K, part, s)
                                  : launch_down<QL_F16>(x, ldx, lora_a, M, K, part, s);
  if (st != QL_OK) return st;
  const int64_t kps = down_k_per_split(K);
  const SkinnyArgs p{(const uint16_t*)x, ldx, packed, absmax, code2, absmax2, nf4_table, offset,
                     log2_bs, log2_bs2, nullptr, nullptr, 0, 0, 0, part, lora_b,
                     (int)((K + kps - 1) / kps), scaling, (uint16_t*)C, ldc, (const uint16_t*)bias,
                     M, N, K, 1.0f};
  if (dtype == QL_BF16)
    return nested ? launch_rows<QL_BF16, true>(p, s) : launch_rows<QL_BF16, false>(p, s);
  return nested ? launch_rows<QL_F16, true>(p, s) : launch_rows<QL_F16, false>(p, s);
}
