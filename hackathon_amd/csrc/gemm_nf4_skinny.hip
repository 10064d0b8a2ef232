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
                     (int)K2, (uint16_t*)C, ldc, (const uint16_t*)bias, M, N, K, alpha};
  if (in_dtype == QL_BF16)
    return nested ? launch_rows<QL_BF16, true>(p, s) : launch_rows<QL_BF16, false>(p, s);
  return nested ? launch_rows<QL_F16, true>(p, s) : launch_rows<QL_F16, false>(p, s);
}
