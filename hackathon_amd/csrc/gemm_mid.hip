// The NT GEMM for outputs that are too few 256 x 256 tiles to fill the chip, for gfx950:
//
//   C[M,N] = alpha * (A B^T + A2 B2^T) (+ bias[n]) (+ residual)
//
// with the operands, segments, rounding and split-K of gemm_nt.hip (which chooses between the
// kernels and sums the partials of a split K), in tiles of 128 x 128, 64 x 128 or 128 x 256. An
// element is the same sum in the same order as there: the second segment's steps first, then the
// split's k upwards.
//
// What bounds it. A wave of a 128 x 128 tile owns 64 x 64: per 64-k step the workgroup reads
// 64 KiB of fragments from LDS and fills 32 KiB, 768 cycles of LDS against 512 of products. So the
// tile runs at half the rate of the 256 x 256 one where that one fills the chip, and pays where it
// does not: 1001 x 3584 x 3584 is 56 tiles of 256 x 256, and splitting K to reach 256 workgroups
// costs a partial tile per workgroup and a second launch, 56 us; 224 tiles of 128 x 128 take
// 33 us unsplit (without its loads the loop takes 25 us, without its products 27).
// - Fragments of the next half step are read while this half's products issue (reads early in the
//   half, so the barrier does not wait for them); the loads of step k + S go out after the barrier
//   of step k, one behind each product, into the buffer that barrier freed.
// - S stages: 4 x 32 KiB for 128 x 128 (41.9 us with 2, one workgroup per CU either way at 224
//   tiles), 3 x 48 KiB for 128 x 256, 3 x 24 KiB and two workgroups per CU for 64 x 128. A step
//   lasts 0.4 us; loads that miss L2 take over one.
// - Every lane keeps its row's 32-bit offset for each of its loads, clamped to the last row, so
//   ragged and aligned operands run the same loop.
#include <utility>

#include "gemm_nt.h"
#include "ql_vec.h"

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

constexpr int BK = 64;
constexpr int kRowBytes = BK * 2;
constexpr int kThreads = 256;
constexpr int kGroupM = 8;

template <int DT> QL_DEV f32x16_t mfma(const uint4& a, const uint4& b, f32x16_t c);
template <> QL_DEV f32x16_t mfma<QL_BF16>(const uint4& a, const uint4& b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                  __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <> QL_DEV f32x16_t mfma<QL_F16>(const uint4& a, const uint4& b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                 __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// 16 B per lane straight into LDS (64 lanes: 1 KiB at LDS offset lds + IMM), hidden from the
// compiler's wait-count pass, which would otherwise drain every load before any LDS read; the K
// loop counts them itself. One wait state separates a write of M0 from the load that reads it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is clobbered on purpose
template <int IMM> QL_DEV void dma(const char* sbase, uint32_t voff, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(sbase), "s"(lds), "n"(IMM)
               : "memory", "m0", "scc");
}
#pragma clang diagnostic pop

// f(integral constants 0 .. N - 1)
template <typename F, int... I>
QL_DEV void unrolled_seq(const F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> QL_DEV void unrolled(const F& f) {
  unrolled_seq(f, std::make_integer_sequence<int, N>{});
}

// Waves WM x WN, each BI x BJ blocks of 32 x 32.
template <int WM_, int WN_, int BI_, int BJ_> struct Tile {
  static constexpr int WM = WM_, WN = WN_, BI = BI_, BJ = BJ_;
  static constexpr int BM = WM * BI * 32, BN = WN * BJ * 32;
  static constexpr int GA = BM / 32, GB = BN / 32;  // DMA instructions per wave and stage
  static constexpr int kStage = (BM + BN) * kRowBytes;
};

// Byte offset of this lane's 16 B for DMA instruction j of an operand tile, from the tile's
// first row: row 8 (4 j + wave) + lane / 8, clamped to the operand's last row, physical chunk
// lane % 8 holding logical chunk (lane % 8) ^ s(row), s as in gemm_nt.hip.
QL_DEV uint32_t dma_off(int j, int wave, int lane, int64_t row0, int64_t rows, int64_t ld) {
  const int r = 8 * (4 * j + wave) + (lane >> 3);
  const int64_t rr = row0 + r < rows ? r : rows - 1 - row0;
  const int c = (lane & 7) ^ (((r >> 1) & 3) | ((r >> 3) & 1) << 2);
  return (uint32_t)(rr * ld * 2 + c * 16);
}

template <int IT, int OT, bool PARTIAL, typename T, int S, int WAVES_EU>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(WAVES_EU, WAVES_EU)))
void gemm_mid_kernel(const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ B,
                     int64_t ldb, const uint16_t* __restrict__ A2, int64_t lda2,
                     const uint16_t* __restrict__ B2, int64_t ldb2, int64_t K2,
                     typename Elem<OT>::T* __restrict__ C, int64_t ldc, float* __restrict__ ws,
                     const uint16_t* __restrict__ bias, int64_t M, int64_t N, int64_t K,
                     int64_t k_per_split, float alpha, const uint16_t* __restrict__ res,
                     int64_t ldr) {
#pragma clang fp contract(off)
  constexpr int BM = T::BM, BN = T::BN, BI = T::BI, BJ = T::BJ, GA = T::GA, GB = T::GB;
  constexpr int kOutBytes = BM * BN * (PARTIAL || OT == QL_F32 ? 4 : 2);
  constexpr int kLds = S * T::kStage > kOutBytes ? S * T::kStage : kOutBytes;
  __shared__ __attribute__((aligned(1024))) char smem[kLds];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / T::WN, wn = wave % T::WN;

  // tile of this workgroup: XCD-contiguous renumbering, then groups of kGroupM tile rows
  int64_t m0, n0;
  {
    const int64_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int64_t total = tiles_m * tiles_n, t = blockIdx.x;
    const int64_t q = total / 8, r = total % 8, xcd = t % 8;
    const int64_t tt = xcd * q + (xcd < r ? xcd : r) + t / 8;
    const int64_t g = tt / (kGroupM * tiles_n), first = g * kGroupM;
    const int64_t gm = tiles_m - first < kGroupM ? tiles_m - first : kGroupM;
    const int64_t in = tt - g * kGroupM * tiles_n;
    m0 = (first + in % gm) * BM;
    n0 = (in / gm) * BN;
  }
  const int64_t kb = (int64_t)blockIdx.y * k_per_split;
  const int64_t ke = kb + k_per_split < K ? kb + k_per_split : K;
  // steps: the second segment's first (last split only), then this split's range of the first
  const int nk2 = (int)blockIdx.y == (int)gridDim.y - 1 ? (int)(K2 / BK) : 0;
  const int nk = nk2 + (int)((ke - kb) / BK);

  uint32_t oa[GA], ob[GB];
#pragma unroll
  for (int j = 0; j < GA; ++j) oa[j] = dma_off(j, wave, lane, m0, M, lda);
#pragma unroll
  for (int j = 0; j < GB; ++j) ob[j] = dma_off(j, wave, lane, n0, N, ldb);
  const char* a0 = reinterpret_cast<const char*>(A + m0 * lda + kb);
  const char* b0 = reinterpret_cast<const char*>(B + n0 * ldb + kb);

  // DMA instruction j (A's first) of step t into `stage`; past the end the last step again, so
  // that the counts hold
  struct Src {
    const char *a, *b;
    bool second;
  };
  auto source = [&](int t) {
    t = t < nk ? t : nk - 1;
    if (t < nk2)
      return Src{reinterpret_cast<const char*>(A2 + m0 * lda2 + (int64_t)t * BK),
                 reinterpret_cast<const char*>(B2 + n0 * ldb2 + (int64_t)t * BK), true};
    const int64_t k = (int64_t)(t - nk2) * kRowBytes;
    return Src{a0 + k, b0 + k, false};
  };

  f32x16_t acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) acc[i][j] = f32x16_t{};

  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)smem) +
                        1024u * (uint32_t)wave;
#pragma unroll
  for (int t = 0; t < S; ++t) {
    const Src src = source(t);
    const uint32_t stage = lds0 + (uint32_t)(t * T::kStage);
    unrolled<GA>([&](auto j) {
      dma<4096 * j.value>(src.a, src.second ? dma_off(j.value, wave, lane, m0, M, lda2) : oa[j.value], stage);
    });
    unrolled<GB>([&](auto j) {
      dma<BM * kRowBytes + 4096 * j.value>(
          src.b, src.second ? dma_off(j.value, wave, lane, n0, N, ldb2) : ob[j.value], stage);
    });
  }

  const int r = lane & 31;
  const int swz = ((r >> 1) & 3) | ((r >> 3) & 1) << 2;
  const int a_off = (wm * BI * 32 + r) * kRowBytes;
  const int b_off = BM * kRowBytes + (wn * BJ * 32 + r) * kRowBytes;
  constexpr int RH = 2 * (BI + BJ), MF = 2 * BI * BJ, G = GA + GB;
  // fragment e of a half: A blocks then B blocks of its first 16 k, then of its second
  uint4 f0[RH], f1[RH];
  auto read = [&](const char* stage, int half, int e) {
    const int kk = e / (BI + BJ), b = e % (BI + BJ);
    const int c = ((half * 4 + kk * 2 + (lane >> 5)) ^ swz) * 16;
    return *reinterpret_cast<const uint4*>(
        stage + c + (b < BI ? a_off + b * 32 * kRowBytes : b_off + (b - BI) * 32 * kRowBytes));
  };
  auto product = [&](const uint4 (&f)[RH], int e) {
    const int kk = e / (BI * BJ), i = e % (BI * BJ) / BJ, j = e % BJ;
    acc[i][j] = mfma<IT>(f[kk * (BI + BJ) + BI + j], f[kk * (BI + BJ) + i], acc[i][j]);
  };
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 1) * G) : "memory");
#pragma unroll
  for (int e = 0; e < RH; ++e) f0[e] = read(smem, 0, e);
  int cur = 0;
  for (int kt = 0; kt < nk; ++kt) {
    const int nxt = cur + 1 == S ? 0 : cur + 1;
    const char* cs = smem + cur * T::kStage;
    const char* ns = smem + nxt * T::kStage;
    // first half: its products, and the second half's fragments (in the first half of them)
    constexpr int RS = (MF + 1) / 2;
    unrolled<MF>([&](auto e) {
#pragma unroll
      for (int q = e.value * RH / RS; q < (e.value + 1) * RH / RS && q < RH; ++q)
        f1[q] = read(cs, 1, q);
      product(f0, e.value);
      __builtin_amdgcn_sched_barrier(0);
    });
    // this wave's share of step kt + 1 has landed (S - 2 later steps may be in flight) and it has
    // read all of step kt; past the barrier that holds for every wave: step kt + 1 may be read
    // and step kt's buffer refilled with step kt + S
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * G) : "memory");
    const Src src = source(kt + S);
    const uint32_t stage = lds0 + (uint32_t)(cur * T::kStage);
    unrolled<MF>([&](auto e) {
      constexpr int q0 = e.value * G / MF, q1 = (e.value + 1) * G / MF;
      unrolled<q1 - q0>([&](auto dq) {
        constexpr int q = q0 + dq.value;
        if constexpr (q < GA) dma<4096 * q>(src.a, oa[q], stage);
        else dma<BM * kRowBytes + 4096 * (q - GA)>(src.b, ob[q - GA], stage);
      });
#pragma unroll
      for (int q = e.value * RH / MF; q < (e.value + 1) * RH / MF; ++q) f0[q] = read(ns, 0, q);
      product(f1, e.value);
      __builtin_amdgcn_sched_barrier(0);
    });
    cur = nxt;
  }
  // the clamped loads past the end still write LDS: they land before the tile goes through it
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // The tile leaves through LDS, whole rows at a time (4 consecutive columns of 32 rows per
  // register group would store 8 or 16 B pieces of 32 rows per instruction).
  if constexpr (PARTIAL || OT == QL_F32) {
    constexpr int kRow = BN * 4, kSwz = BN / 4 - 1 < 31 ? BN / 4 - 1 : 31;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int tr = (wm * BI + i) * 32 + r;
          const int c = (wn * BJ + j) * 32 + 8 * g + 4 * (lane >> 5);
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = acc[i][j][4 * g + e];
            if constexpr (!PARTIAL) {
              v[e] = alpha * v[e];
              if (bias && n0 + c + e < N) v[e] += Elem<IT>::to_f32(bias[n0 + c + e]);
            }
          }
          *reinterpret_cast<float4*>(smem + tr * kRow + (((c >> 2) ^ (tr & kSwz)) << 4)) =
              make_float4(v[0], v[1], v[2], v[3]);
        }
    __syncthreads();
    constexpr int kChunks = BN / 4;
    float* out = PARTIAL ? ws + (int64_t)blockIdx.y * M * N : reinterpret_cast<float*>(C);
    const int64_t ldo = PARTIAL ? N : ldc;
    const bool vec = (ldo & 3) == 0 && ((uintptr_t)out & 15) == 0;
    for (int idx = threadIdx.x; idx < BM * kChunks; idx += kThreads) {
      const int tr = idx / kChunks, q = idx % kChunks;
      const int64_t row = m0 + tr, col = n0 + 4 * q;
      if (row >= M || col >= N) continue;
      const float4 v = *reinterpret_cast<const float4*>(smem + tr * kRow + ((q ^ (tr & kSwz)) << 4));
      float* cp = out + row * ldo + col;
      if (vec && col + 4 <= N) {
        *reinterpret_cast<float4*>(cp) = v;
      } else {
        const float w[4] = {v.x, v.y, v.z, v.w};
        for (int e = 0; e < 4 && col + e < N; ++e) cp[e] = w[e];
      }
    }
  } else {
    constexpr int kRow = BN * 2, kChunks = BN / 8, kSwz = kChunks - 1 < 15 ? kChunks - 1 : 15;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int tr = (wm * BI + i) * 32 + r;
          const int c = (wn * BJ + j) * 32 + 8 * g + 4 * (lane >> 5);
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = alpha * acc[i][j][4 * g + e];
            if (bias && n0 + c + e < N) v[e] += Elem<IT>::to_f32(bias[n0 + c + e]);
          }
          const uint2 w = OT == QL_BF16
                              ? make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]))
                              : make_uint2(pack_f16x2(v[0], v[1]), pack_f16x2(v[2], v[3]));
          *reinterpret_cast<uint2*>(smem + tr * kRow + (((c >> 3) ^ (tr & kSwz)) << 4) + (c & 4) * 2) = w;
        }
    __syncthreads();
    const bool vec = (ldc & 7) == 0 && ((uintptr_t)C & 15) == 0;
    for (int idx = threadIdx.x; idx < BM * kChunks; idx += kThreads) {
      const int tr = idx / kChunks, q = idx % kChunks;
      const int64_t row = m0 + tr, col = n0 + 8 * q;
      if (row >= M || col >= N) continue;
      uint4 v = *reinterpret_cast<const uint4*>(smem + tr * kRow + ((q ^ (tr & kSwz)) << 4));
      auto* cp = C + row * ldc + col;
      if (vec && col + 8 <= N) {
        if (res) {  // the rounded product plus the residual, rounded again
          float pv[8], rv[8];
          Vec8<OT>::unpack(v, pv);
          Vec8<OT>::unpack(*reinterpret_cast<const uint4*>(res + row * ldr + col), rv);
#pragma unroll
          for (int e = 0; e < 8; ++e) pv[e] = pv[e] + rv[e];
          v = Vec8<OT>::pack(pv);
        }
        *reinterpret_cast<uint4*>(cp) = v;
      } else {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        for (int e = 0; e < 8 && col + e < N; ++e) {
          uint16_t o = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
          if (res)
            o = Elem<OT>::from_f32(Elem<OT>::to_f32(o) + Elem<OT>::to_f32(res[row * ldr + col + e]));
          cp[e] = o;
        }
      }
    }
  }
}

struct Args {
  const void *A, *B, *A2, *B2, *bias, *res;
  int64_t lda, ldb, lda2, ldb2, ldc, ldr, M, N, K, K2;
  void* C;
  float* ws;
  float alpha;
  int64_t k_per_split;
  int splits;
};

template <int IT, int OT, typename T, int S, int W>
int launch(const Args& p, hipStream_t s) {
  const int64_t tiles = ((p.M + T::BM - 1) / T::BM) * ((p.N + T::BN - 1) / T::BN);
  if (p.splits <= 1) {
    hipLaunchKernelGGL((gemm_mid_kernel<IT, OT, false, T, S, W>), dim3((unsigned)tiles, 1),
                       dim3(kThreads), 0, s, (const uint16_t*)p.A, p.lda, (const uint16_t*)p.B,
                       p.ldb, (const uint16_t*)p.A2, p.lda2, (const uint16_t*)p.B2, p.ldb2, p.K2,
                       (typename Elem<OT>::T*)p.C, p.ldc, nullptr, (const uint16_t*)p.bias, p.M,
                       p.N, p.K, p.K, p.alpha, (const uint16_t*)p.res, p.ldr);
    return ql_launch_status();
  }
  hipLaunchKernelGGL((gemm_mid_kernel<IT, QL_F32, true, T, S, W>),
                     dim3((unsigned)tiles, (unsigned)p.splits), dim3(kThreads), 0, s,
                     (const uint16_t*)p.A, p.lda, (const uint16_t*)p.B, p.ldb,
                     (const uint16_t*)p.A2, p.lda2, (const uint16_t*)p.B2, p.ldb2, p.K2,
                     (float*)nullptr, (int64_t)0, p.ws, (const uint16_t*)nullptr, p.M, p.N, p.K,
                     p.k_per_split, 1.0f, (const uint16_t*)nullptr, (int64_t)0);
  return ql_launch_status();
}

template <int IT, int OT>
int launch_tile(QlGemmTile tile, const Args& p, hipStream_t s) {
  switch (tile) {
    case QlGemmTile::k128x128: return launch<IT, OT, Tile<2, 2, 2, 2>, 4, 1>(p, s);
    case QlGemmTile::k64x128: return launch<IT, OT, Tile<2, 2, 1, 2>, 3, 2>(p, s);
    case QlGemmTile::k128x256: return launch<IT, OT, Tile<2, 2, 2, 4>, 3, 1>(p, s);
    default: return QL_EINVAL;
  }
}

}  // namespace

int ql_gemm_mid(QlGemmTile tile, int in_dtype, int c_dtype, int64_t M, int64_t N, int64_t K,
                const void* A, int64_t lda, const void* B, int64_t ldb, const void* A2,
                int64_t lda2, const void* B2, int64_t ldb2, int64_t K2, void* C, int64_t ldc,
                const void* bias, float alpha, int64_t k_per_split, int splits, float* ws,
                hipStream_t s, const void* residual, int64_t ld_residual) {
  const Args p{A,   B,  A2, B2, bias, residual, lda, ldb,   lda2,        ldb2,  ldc, ld_residual,
               M,   N,  K,  K2, C,    ws,       alpha, k_per_split, splits};
  if (in_dtype == QL_BF16) {
    QL_DISPATCH_DTYPE(c_dtype, OT, return (launch_tile<QL_BF16, OT>(tile, p, s)));
  } else if (in_dtype == QL_F16) {
    QL_DISPATCH_DTYPE(c_dtype, OT, return (launch_tile<QL_F16, OT>(tile, p, s)));
  }
  return QL_EDTYPE;
}
