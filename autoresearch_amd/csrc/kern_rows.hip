// kern_rows.hip -- MFMA GEMM for few token rows (batched decode, prompt
// chunks, short prefills) on gfx950: C[M][N] = epi(s_m * (A[M][K] . W[N][K]^T)),
// the operands, precision and epilogues of k_gemm (kern_gemm.hip).
//
// At these sizes a linear is bound by latency: the weights (1-8 MB) stream in
// about a microsecond, a launch costs 2-3, and an LDS pipeline walks K in a
// serial chain of stage hand-overs. So nothing is staged: a block owns a
// (16 TM) x (16 TN) tile, its 8 wavefronts take one eighth of K each, and
// every wavefront loads its A and W fragments from memory straight into MFMA
// operand registers (v_mfma_f32_16x16x32: a 1 KB operand tile is one load),
// U steps in flight.
// The 8 partial tiles meet in LDS, are added in wavefront order and go through
// the epilogue in the same launch: no split-K scratch and no reduce kernel.
// What bounds it then is what one CU can take in (~20 bytes a clock from
// row-major operands, twice that from operand tiles (tile_at), whose loads
// are consecutive) and the launch itself. Measured at d_model 768, us a
// launch over 12 layers' weights (the split-K GEMM and reduce kernel it
// replaced in front): M = 64 QKV 11.5 -> 5.7, proj 7.8 -> 3.5, fc 11.0 ->
// 4.5, proj2 9.3 -> 5.3; M = 7 8.3 -> 4.0, 6.8 -> 3.4, 8.2 -> 3.9, 7.9 -> 5.4;
// M = 150 in fp16 against 64x64 LDS tiles 10.2 -> 5.9, 7.8 -> 3.5, 9.5 -> 4.8,
// 17.7 -> 5.4.
// Which wavefront takes which K range depends on K alone, so a row's products
// are summed in the same order on every tile. The row norm is not: RESID leaves
// one sum of squares per tile of columns, and those are added 512 / (16 TM)
// threads at a time, so the row count of the pass, which picks the tile, moves
// the last bits of a row.
#include "fgpt_internal.h"
#include "kern_common.h"
#include "kern_epi.h"

namespace fgpt {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int RW = 8, RNT = 64 * RW;  // wavefronts (K ranges) and threads of a block
constexpr int RKS = 32;               // K of one MFMA step

template <bool P16>
__device__ __forceinline__ f32x4_t mma_16x16(const uint4& a, const uint4& b, const f32x4_t& c) {
  if constexpr (P16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Sum over the LW lanes that hold one row of the tile (8, 16 or 32 adjacent
// lanes of a wavefront), the same value in each of them.
template <int LW>
__device__ __forceinline__ float row_sum(float v) {
  if constexpr (LW == 32) return half_sum(v);
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  v += dpp_f<0x141>(v);
  if constexpr (LW == 16) v += dpp_f<0x140>(v);
  return v;
}

template <int EPI, int TM, int TN, int U, bool P16>
__global__ __launch_bounds__(RNT) void k_gemm_rows(GemvArgs a, const int32_t* __restrict__ d_pos) {
  constexpr int BM = 16 * TM, BN = 16 * TN, AP = P16 ? 1 : 2;
  constexpr int STR = BN + 4;                              // floats per partial-tile row in LDS
  constexpr int PAIRS = BM * BN / 2, PPT = (PAIRS + RNT - 1) / RNT;  // column pairs per thread
  constexpr int SP = RNT / BM, SQ = 128 / SP;              // threads per row, partials per thread
  __shared__ float red[RW * BM * STR];
  __shared__ float sinv[BM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = a.M, N = a.N, K = a.K;
  // Blocks go to the 8 XCDs round-robin by linear id: the row tiles of one
  // column tile run on one XCD, so each weight row enters one L2.
  const int mt = gridDim.y, nt = gridDim.x;
  const int lin = blockIdx.x + nt * blockIdx.y;
  int tn, tm;
  if ((nt & 7) == 0) {
    const int i = lin >> 3;
    tn = (lin & 7) + 8 * (i / mt);
    tm = i % mt;
  } else {
    tn = lin % nt;
    tm = lin / nt;
  }
  const int m0 = tm * BM, n0 = tn * BN;

  const uint16_t* ap[TM];
  const uint16_t* wp[TN];
  // rows past M repeat the last one (never stored): their lanes ask for lines
  // that others ask for, so a block of 7 rows takes in half of each A tile (16
  // decode steps of 7 sequences 6459 -> 6031 us)
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int rb = min((m0 >> 4) + i, (M - 1) >> 4), r = min(lane & 15, M - 1 - 16 * rb);
    ap[i] = a.xs + (int64_t)rb * K * 16 + (lane >> 4) * 128 + r * 8;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j)
    wp[j] = a.w + (int64_t)((n0 >> 4) + j) * K * 16 + lane * 8;

  const int S = K / RKS, s0 = wv * S / RW, n = (wv + 1) * S / RW - s0;
  uint4 fh[U][TM], fl[U][TM], fw[U][TN];
  auto load = [&](int u, int i) {  // step i of this wavefront (past the end: the last, unused)
    const int64_t k = (int64_t)min(s0 + min(i, n - 1), S - 1) * (RKS * 16);
#pragma unroll
    for (int j = 0; j < TN; ++j) fw[u][j] = *reinterpret_cast<const uint4*>(wp[j] + k);
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      fh[u][t] = *reinterpret_cast<const uint4*>(ap[t] + k);
      if constexpr (AP == 2) fl[u][t] = *reinterpret_cast<const uint4*>(ap[t] + a.xs_plane + k);
    }
  };
  if (n > 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, u);
  }

  // the epilogue's operands, requested behind the first fragments: the row
  // norm's partial sums, RoPE coefficients, the residual
  float sq[SQ];
  if (a.norm) {
    const int r = tid / SP, p = tid % SP;
    const float* sp = a.ssq_in + (int64_t)min(m0 + r, M - 1) * a.ssq_n;
#pragma unroll
    for (int k = 0; k < SQ; ++k) sq[k] = p + k * SP < a.ssq_n ? sp[p + k * SP] : 0.f;
  }
  const int pos0 = d_pos ? *d_pos : a.pos0;
  float e0[PPT], e1[PPT];
#pragma unroll
  for (int k = 0; k < PPT; ++k) {
    const int e = tid + k * RNT, m = m0 + e / (BN / 2), c = n0 + 2 * (e % (BN / 2));
    e0[k] = e1[k] = 0.f;
    if (e < PAIRS && m < M) {
      if constexpr (EPI == GV_QKV) qkv_pair_coeffs(a, m, pos0, c, e0[k], e1[k]);
      if constexpr (EPI == GV_RESID) {
        const float2 x = *reinterpret_cast<const float2*>(a.y + (int64_t)m * N + c);
        e0[k] = x.x;
        e1[k] = x.y;
      }
    }
  }

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < n; i += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i + u < n) {
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[t][j] = mma_16x16<P16>(fh[u][t], fw[u][j], acc[t][j]);
        if constexpr (AP == 2) {
#pragma unroll
          for (int t = 0; t < TM; ++t)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[t][j] = mma_16x16<P16>(fl[u][t], fw[u][j], acc[t][j]);
        }
        if (i + U < n) load(u, i + u + U);
      }
    }
  }
  // lane l holds column l % 16 of rows 4 (l / 16) .. + 3 of a 16x16 block
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[(wv * BM + 16 * i + 4 * (lane >> 4) + r) * STR + 16 * j + (lane & 15)] = acc[i][j][r];
  if (a.norm) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < SQ; ++k) s += sq[k];
    for (int k = tid % SP + SQ * SP; k < a.ssq_n; k += SP)  // (more than 128 partials: d_model > 2048)
      s += a.ssq_in[(int64_t)min(m0 + tid / SP, M - 1) * a.ssq_n + k];
    s = SP == 8 ? row_sum<8>(s) : SP == 16 ? row_sum<16>(s) : row_sum<32>(s);
    if (tid % SP == 0) sinv[tid / SP] = 1.0f / sqrtf(s / (float)K + a.eps);
  }
  __syncthreads();

#pragma unroll
  for (int k = 0; k < PPT; ++k) {
    const int e = tid + k * RNT;
    if (PAIRS % RNT != 0 && e >= PAIRS) break;  // (whole wavefronts: 64 divides PAIRS)
    const int ml = e / (BN / 2), cl = 2 * (e % (BN / 2)), m = m0 + ml, c = n0 + cl;
    const bool live = m < M;
    float v0 = 0.f, v1 = 0.f;
#pragma unroll
    for (int w = 0; w < RW; ++w) {  // wavefront order
      const float2 p = *reinterpret_cast<const float2*>(red + (w * BM + ml) * STR + cl);
      v0 += p.x;
      v1 += p.y;
    }
    if constexpr (P16) {  // (the weights were stored scaled by 1 / wscale, a power of 2)
      v0 *= a.wscale;
      v1 *= a.wscale;
    }
    if (a.norm) {
      v0 *= sinv[ml];
      v1 *= sinv[ml];
    }
    const int64_t o = (int64_t)m * N + c;
    if constexpr (EPI == GV_QKV) {
      if (live) qkv_pair_store<P16>(a, m, pos0, c, v0, v1, e0[k], e1[k]);
    } else if constexpr (EPI == GV_RESID) {
      float x0 = 0.f, x1 = 0.f;
      if (live) {
        x0 = e0[k] + v0;
        x1 = e1[k] + v1;
        *reinterpret_cast<float2*>(a.y + o) = make_float2(x0, x1);
        f16_guard<P16>(a, x0);
        f16_guard<P16>(a, x1);
        put2<P16>(x0, x1, a.ys + tile_at(m, c, N), a.ys_plane);
      }
      const float s = row_sum<BN / 2>(x0 * x0 + x1 * x1);
      if (live && cl == 0) a.ssq_out[(int64_t)m * nt + tn] = s;
    } else if constexpr (EPI == GV_RELU2) {
      if (live) {
        const float t0 = v0 < 0.f ? 0.f : v0, t1 = v1 < 0.f ? 0.f : v1;
        f16_guard<P16>(a, t0 * t0);
        f16_guard<P16>(a, t1 * t1);
        put2<P16>(t0 * t0, t1 * t1, a.ys + tile_at(m, c, N), a.ys_plane);
      }
    } else {
      if (live) *reinterpret_cast<float2*>(a.y + o) = make_float2(v0, v1);
    }
  }
}

template <int EPI, int TM, int TN, int U, bool P16>
void launch_rows_tile(hipStream_t s, const GemvArgs& a, const int32_t* d_pos) {
  const dim3 g((unsigned)(a.N / (16 * TN)), (unsigned)((a.M + 16 * TM - 1) / (16 * TM)));
  FG_LAUNCH((k_gemm_rows<EPI, TM, TN, U, P16>), g, dim3(RNT), 0, s, a, d_pos);
}

template <int EPI, bool P16>
void launch_rows_epi(hipStream_t s, const GemvArgs& a, const int32_t* d_pos) {
  const RowsTile t = gemm_rows_tile(a.M, a.N);
  if (t.tm == 4) launch_rows_tile<EPI, 4, 4, 2, P16>(s, a, d_pos);
  else if (t.tn == 4) launch_rows_tile<EPI, 2, 4, 3, P16>(s, a, d_pos);
  else if (t.tm == 2) launch_rows_tile<EPI, 2, 2, 4, P16>(s, a, d_pos);
  else if (t.tn == 2) launch_rows_tile<EPI, 1, 2, 6, P16>(s, a, d_pos);
  else launch_rows_tile<EPI, 1, 1, 6, P16>(s, a, d_pos);
}

template <bool P16>
void launch_rows_p(hipStream_t s, GemvEpi epi, const GemvArgs& a, const int32_t* d_pos) {
  switch (epi) {
    case GV_QKV: launch_rows_epi<GV_QKV, P16>(s, a, d_pos); break;
    case GV_RESID: launch_rows_epi<GV_RESID, P16>(s, a, d_pos); break;
    case GV_RELU2: launch_rows_epi<GV_RELU2, P16>(s, a, d_pos); break;
    default: launch_rows_epi<GV_STORE, P16>(s, a, d_pos); break;
  }
}

// dst[tile_at(n, k)] = src[n][k]: a workgroup per 16 rows, a thread per
// 16-byte chunk (its stores consecutive).
__global__ __launch_bounds__(256) void k_tile_weights(const bf16_t* __restrict__ src,
                                                      bf16_t* __restrict__ dst, int K) {
  const int64_t blk = (int64_t)blockIdx.x * 16 * K;
  for (int e = threadIdx.x; e < 2 * K; e += 256) {
    const int r = e & 15, k = 8 * (e >> 4);
    *reinterpret_cast<uint4*>(dst + blk + 8 * e) =
        *reinterpret_cast<const uint4*>(src + blk + (int64_t)r * K + k);
  }
}

}  // namespace

// Token rows up to ROWS_MAX_M run here, each GEMM on the smallest tile whose
// blocks fit the CUs in one round (a CU takes in the operands of its tiles at
// a fixed rate, so work spread over every CU and done once is the fastest;
// past one round the next larger tile moves fewer bytes: M = 64, N = 3072 on
// 192 blocks of 32x32 4.5 us, on 384 of 16x32 5.9, on 96 of 32x64 5.0).
RowsTile gemm_rows_tile(int64_t M, int N) {
  if (M > ROWS_MAX_M) return {0, 0};
  static const RowsTile tiles[] = {{1, 1}, {1, 2}, {2, 2}, {2, 4}, {4, 4}};
  for (const RowsTile& t : tiles) {
    if (N % (16 * t.tn) != 0) continue;
    if (((M + 16 * t.tm - 1) / (16 * t.tm)) * (N / (16 * t.tn)) <= cu_count()) return t;
  }
  return {4, 4};
}

void launch_gemm_rows(hipStream_t s, GemvEpi epi, const GemvArgs& a, const int32_t* d_pos) {
  if (a.f16)
    launch_rows_p<true>(s, epi, a, d_pos);
  else
    launch_rows_p<false>(s, epi, a, d_pos);
}

void launch_tile_weights(hipStream_t s, const bf16_t* src, bf16_t* dst, int64_t N, int K) {
  FG_LAUNCH(k_tile_weights, dim3((unsigned)(N / 16)), dim3(256), 0, s, src, dst, K);
}

}  // namespace fgpt
