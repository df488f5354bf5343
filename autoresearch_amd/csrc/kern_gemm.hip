// kern_gemm.hip -- MFMA GEMM for more than 256 token rows (gfx950; fewer run in
// kern_rows.hip).
//
// C[M][N] = epi( s_m * (A[M][K] . W[N][K]^T) ), the y = x W^T of
// linear3d_sgemm (src/lib/fortran_blas.f90:39-57) with rmsnorm0's row scale
// s_m = 1/sqrt(mean(A_m^2) + eps) (src/lib/fortran_rmsnorm.f90:40-60) applied
// to the output rows when `norm` is set (rmsnorm is a per-row scale, so
// norm(x) W^T = s * (x W^T)).
//
// Precision: W is bf16 and exact (the weights are bf16-representable). A is
// an fp32 activation carried as two bf16 terms, A = hi + lo with
// hi = bf16(A), lo = bf16(A - hi), written in that form once by the kernel
// that produced it; both terms go through v_mfma_f32_32x32x16_bf16 with
// fp32 accumulation, so each product carries ~16 mantissa bits of A instead
// of 8. A single bf16 term moves depth-12 logits by ~3e-3 of max|logit|,
// more than the 2e-3 parity bound; the split keeps it ~5e-6. The row norm
// comes from per-row sums of squares of the fp32 values, also written by
// the producer (one partial per producer N tile, summed here in order).
//
// Pipeline: NST stages of BK-wide K slices (BK = 32 or 64) in LDS,
// filled by global_load_lds_dwordx4 (memory -> LDS without registers),
// NST-1 slices in flight while the MFMAs consume the oldest. Both operands
// are stored in 1 KB tiles of 16 rows x 32 K (tile_at), so each DMA reads 1 KB
// of consecutive memory and a stage is a list of tiles: the MFMA operand
// reads (32 rows x one 16-byte chunk per half-wavefront) are two runs of 256
// consecutive bytes, free of bank conflicts without a swizzle.
// Tiling: BM x BN per block of NWM x NWN 64-wide wavefronts, each owning
// (BM/NWM) x (BN/NWN) as 32x32 MFMA blocks, times KG groups of such
// wavefronts that split each slice's K steps between them. The epilogue is
// staged through LDS 64 rows at a time so each thread owns a column pair
// (coalesced stores; a QKV rotation pair in one thread). The host picks the
// tile per shape (launch_tile) so that one round of tiles covers the CUs.
#include <algorithm>

#include "fgpt_internal.h"
#include "kern_common.h"
#include "kern_epi.h"

namespace fgpt {
// Epilogue outputs written streaming (no cache allocation): the ReLU^2 planes
// and the residual (fp32 and planes) are read only by later kernels, from
// other XCDs' L2 mostly, and are too large to stay cached for them (25 MB
// for fc at T=2048); measured ~2.5 us faster per fc and ~0.7 us per residual
// GEMM. QKV's scattered q/k/v stores gained nothing.
constexpr bool NT_RELU2 = true, NT_RESID = true, NT_QKV = false;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// One 32x32x16 MFMA step: bf16 operands, or (P16) fp16 ones.
template <bool P16>
__device__ __forceinline__ f32x16_t mma16(const bf16x8_t& a, const bf16x8_t& b, const f32x16_t& c) {
  if constexpr (P16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

namespace {

// Byte offset within a stage (k tiles of RT row tiles each) of the 16-byte
// chunk c of row r.
template <int RT>
__device__ __forceinline__ int at(int r, int c) {
  return ((c >> 2) * RT + (r >> 4)) * 1024 + ((c & 3) * 16 + (r & 15)) * 16;
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One 64-row pass of the QKV epilogue from the staged tile (fp32 [64][SSTR],
// rows m0 + 64 q ..): q/k/v columns in items of four rotation pairs of one
// row (one wide store per plane and four dims); for tiles holding v columns
// that go to the transposed layout, items of one pair over four consecutive
// rows (positions), so v^T gets one wide store per dim. Rows that do not
// form an aligned run of four positions of one sequence take the per-pair
// path. Every item's RoPE coefficients are loaded before any item stores.
template <int BN, int NT, bool P16>
__device__ __forceinline__ void qkv_tile_pass(const GemvArgs& a, const float* stage,
                                              const float* sinv, int m0, int n0, int q,
                                              bool rows_fast, int pos0) {
  constexpr int SSTR = BN + 4, NI = 8 * BN / NT;  // items per thread (64 * BN / 8 in all)
  static_assert(NI * NT == 8 * BN, "epilogue items / block size mismatch");
  const int tid = threadIdx.x, M = a.M, hd = a.hd, qdk = (a.H + a.KH) * hd;
  if (!rows_fast) {
    float4 c4[NI], s4[NI];
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int e = tid + k * NT, srow = e / (BN / 8), pc = 8 * (e % (BN / 8));
      const int m = m0 + q * 64 + srow, n = n0 + pc;
      c4[k] = s4[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (m < M && n < qdk) {
        const int base = n < a.H * hd ? n : n - a.H * hd;
        const int64_t at = (int64_t)(pos0 + m % a.T) * (hd / 2) + ((base % hd) >> 1);
        c4[k] = *reinterpret_cast<const float4*>(a.cosb + at);
        s4[k] = *reinterpret_cast<const float4*>(a.sinb + at);
      }
    }
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int e = tid + k * NT, srow = e / (BN / 8), pc = 8 * (e % (BN / 8));
      const int ml = q * 64 + srow, m = m0 + ml;
      if (m >= M) continue;
      const float4 lo = *reinterpret_cast<const float4*>(stage + srow * SSTR + pc);
      const float4 hi = *reinterpret_cast<const float4*>(stage + srow * SSTR + pc + 4);
      const float sc = a.norm ? sinv[ml] : 1.f;
      const float x[8] = {lo.x * sc, lo.y * sc, lo.z * sc, lo.w * sc,
                          hi.x * sc, hi.y * sc, hi.z * sc, hi.w * sc};
      qkv_quad_store<NT_QKV, P16>(a, m, pos0, n0 + pc, x, c4[k], s4[k]);
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < NI; ++k) {
    const int e = tid + k * NT, g = e % 16, pc = 2 * (e / 16);
    const int r0 = 4 * g, n = n0 + pc, mb = m0 + q * 64 + r0;
    float x1[4], x2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float sc = a.norm ? sinv[q * 64 + r0 + i] : 1.f;
      x1[i] = stage[(r0 + i) * SSTR + pc] * sc;
      x2[i] = stage[(r0 + i) * SSTR + pc + 1] * sc;
    }
    const int t0 = mb % a.T, pos = pos0 + t0;
    const bool run4 = n >= qdk && a.vt && mb + 3 < M && t0 + 3 < a.T && (pos & 3) == 0;
    if (run4) {
      const int base = n - qdk, head = base / hd, j = (base % hd) >> 1, b = mb / a.T;
      uint16_t* p = a.vt + ((int64_t)b * a.KH + head) * hd * a.npos + pos;
      if (a.kv16) {  // the planes carry what the bf16 cache holds
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x1[i] = kv_val(a, x1[i]);
          x2[i] = kv_val(a, x2[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f16_guard<P16>(a, x1[i]);
        f16_guard<P16>(a, x2[i]);
      }
      put4<P16, NT_QKV>(x1, p + (int64_t)j * a.npos, a.kv_plane);
      put4<P16, NT_QKV>(x2, p + (int64_t)(j + hd / 2) * a.npos, a.kv_plane);
      if (a.vc) {
        const int kd = a.KH * hd;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int64_t v = ((int64_t)b * a.maxT + pos + i) * kd + head * hd;
          kv_put(a, a.vc, v + j, x1[i]);
          kv_put(a, a.vc, v + j + hd / 2, x2[i]);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (mb + i < M) qkv_pair_epilogue<P16>(a, mb + i, pos0, n, x1[i], x2[i]);
    }
  }
}

// KG > 1 splits each stage's 16-deep K steps over KG groups of NWM x NWN
// wavefronts (group g takes steps g, g + KG, ..): a tile too small to give
// every SIMD two wavefronts of its own still keeps them all busy. The
// groups' partial sums meet in the LDS staging buffer in a fixed order
// (KG - 1 first, 0 last), so the result does not depend on timing.
template <int EPI, int BM, int BN, int NWM, int NWN, int BK, int NST, int KG = 1, bool P16 = false>
__global__ __launch_bounds__(64 * NWM * NWN * KG) void k_gemm(GemvArgs a,
                                                             const int32_t* __restrict__ d_pos) {
  constexpr int NWT = NWM * NWN, NW = NWT * KG, NT = 64 * NW;
  constexpr int WM = BM / (32 * NWM), WN = BN / (32 * NWN);  // 32x32 blocks per wave
  // a stage: for each 32 of K the tiles of A hi, A lo and W, one wavefront
  // instruction each
  constexpr int AP = P16 ? 1 : 2;  // operand planes of A (hi and lo, or one fp16)
  constexpr int ROWS = AP * BM + BN, RT = ROWS / 16;
  constexpr int GROUPS = RT * (BK / 32);     // 1 KB tiles per stage
  // groups per wavefront per stage; when NW does not divide GROUPS, the
  // spare slots repeat the last group (the same bytes to the same place)
  constexpr int GPW = (GROUPS + NW - 1) / NW;
  static_assert(WM >= 1 && WN >= 1, "tile / wave grid mismatch");
  static_assert(KG == 1 || (BM == 64 && (BK / 16) % KG == 0), "K groups: one 64-row pass");
  constexpr int STAGE_BYTES = GROUPS * 1024;
  constexpr int SSTR = BN + 4;  // epilogue staging row stride (floats)
  // NST stages of STAGE_BYTES; after the K loop the same memory (sized for
  // the larger of the two) stages the epilogue (the DMA is issued from asm, so the compiler never waits on it
  // for an LDS read: the stage_sync() calls order them)
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  float* stage = reinterpret_cast<float*>(smem);
  __shared__ float sinv[BM];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int kg = wid / NWT, wm = (wid % NWT) / NWN, wn = wid % NWN;
  // Blocks go to the 8 XCDs round-robin by linear id. Remap so that XCD x
  // runs a contiguous run of tiles in row-major order: tiles sharing an A
  // row-block (and the weight panel sweep) stay in one XCD's L2.
  const int nbn = gridDim.x, ntile = gridDim.x * gridDim.y;
  int lin = blockIdx.x + nbn * blockIdx.y;
  if ((ntile & 7) == 0) lin = (lin & 7) * (ntile >> 3) + (lin >> 3);
  const int m0 = (lin / nbn) * BM, n0 = (lin % nbn) * BN;
  const int M = a.M, K = a.K;

  // This lane's source of each of its load groups: chunk `lane` of tile g's
  // 1 KB (row tiles past M repeat the last one and are never stored); a
  // K slice further on is BK / 32 tiles (16 BK elements) away.
  const uint16_t* src[GPW];
#pragma unroll
  for (int q = 0; q < GPW; ++q) {
    const int g = min(wid + NW * q, GROUPS - 1), rt = g % RT, kt = g / RT;
    const uint16_t* base;
    if (rt < AP * (BM / 16)) {  // A hi, then A lo
      const int ar = rt < BM / 16 ? rt : rt - BM / 16;
      base = a.xs + (rt < BM / 16 ? 0 : a.xs_plane) +
             (int64_t)min((m0 >> 4) + ar, (M - 1) >> 4) * K * 16;
    } else {
      base = a.w + (int64_t)((n0 >> 4) + rt - AP * (BM / 16)) * K * 16;
    }
    src[q] = base + kt * 512 + lane * 8;
  }

  // epilogue items (8 columns of one row of a 64-row pass) per thread
  constexpr int ITEMS = 64 * (BN / 8), EPT = (ITEMS + NT - 1) / NT;
  // RESID row sums of squares: one value per item in LDS (sqs, a padded
  // [64][BN / 8] after the staged tile), a row's summed by four threads
  constexpr int SQS = BN / 8 + 1;
  // RESID: the residual tile is read now, so its latency hides behind the
  // K loop instead of stalling the epilogue
  float4 xres[EPI == GV_RESID ? (BM / 64) * EPT : 1][2];
  if (EPI == GV_RESID) {
#pragma unroll
    for (int q = 0; q < BM / 64; ++q)
#pragma unroll
      for (int k = 0; k < EPT; ++k) {
        const int e = min(tid + k * NT, ITEMS - 1), m = min(m0 + q * 64 + e / (BN / 8), M - 1);
        const float4* p = reinterpret_cast<const float4*>(a.y + (int64_t)m * a.N + n0 +
                                                          8 * (e % (BN / 8)));
        xres[q * EPT + k][0] = p[0];
        xres[q * EPT + k][1] = p[1];
      }
  }

  f32x16_t acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nk = K / BK;  // K % BK == 0 (checked by the host)
  const int klast = K - BK;
  uint32_t ldsq[GPW];  // LDS byte offset of each of this wavefront's groups
#pragma unroll
  for (int q = 0; q < GPW; ++q)
    ldsq[q] = __builtin_amdgcn_readfirstlane(lds_off(smem) + min(wid + NW * q, GROUPS - 1) * 1024);
  auto fill = [&](int stg, int k0) {
#pragma unroll
    for (int q = 0; q < GPW; ++q) dma16(src[q] + k0 * 16, ldsq[q] + stg * STAGE_BYTES);
  };
  auto consume = [&](int si) {
    const uint8_t* stg = smem + si * STAGE_BYTES;
#pragma unroll
    for (int k2 = 0; k2 < BK / 16 / KG; ++k2) {
      const int kk = k2 * KG + kg;         // this group's 16-deep step of the stage
      const int c = 2 * kk + (lane >> 5);  // logical chunk of this half-wave
      bf16x8_t ah[WM], al[WM], bw[WN];
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        const int r = (wm * WM + i) * 32 + (lane & 31);
        ah[i] = *(const bf16x8_t*)(stg + at<RT>(r, c));
        if constexpr (!P16) al[i] = *(const bf16x8_t*)(stg + at<RT>(BM + r, c));
      }
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const int r = AP * BM + (wn * WN + j) * 32 + (lane & 31);
        bw[j] = *(const bf16x8_t*)(stg + at<RT>(r, c));
      }
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = mma16<P16>(ah[i], bw[j], acc[i][j]);
      if constexpr (!P16) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j) acc[i][j] = mma16<false>(al[i], bw[j], acc[i][j]);
      }
    }
  };
  // prologue: slices 0 .. NST-2 in flight; then each step waits for its
  // slice and refills the stage consumed one step earlier (NST-1 slices
  // ahead; loads past the end re-read the last slice so the outstanding
  // count is fixed)
#pragma unroll
  for (int si = 0; si < NST - 1; ++si) fill(si, min(si * BK, klast));
  for (int kt = 0; kt < nk; kt += NST) {
#pragma unroll
    for (int si = 0; si < NST; ++si) {
      if (kt + si < nk) {  // uniform; only the last group can be partial
        stage_sync<(NST - 2) * GPW>();
        fill((si + NST - 1) % NST, min((kt + si + NST - 1) * BK, klast));
        consume(si);
      }
    }
  }
  wait_vmcnt<0>();
  __syncthreads();

  // row scale from the producer's partial sums of squares
  if (a.norm) {
    for (int r = tid; r < BM; r += NT) {
      float ssum = 0.f;
      if (m0 + r < M)
        for (int t = 0; t < a.ssq_n; ++t) ssum += a.ssq_in[(int64_t)(m0 + r) * a.ssq_n + t];
      sinv[r] = 1.0f / sqrtf(ssum / (float)K + a.eps);
    }
    __syncthreads();
  }

  // epilogue through LDS, 64 tile rows (two 32-row blocks) per pass
  const int pos0 = d_pos ? *d_pos : a.pos0;
  // Tiles holding v columns that go to the transposed bf16 layout
  // ([..][hd][npos]: positions contiguous) walk the staged tile row-fastest,
  // so a wavefront's stores cover 64 consecutive positions of one dim.
  const bool rows_fast = EPI == GV_QKV && a.vt && n0 + BN > (a.H + a.KH) * a.hd;
  float* sqs = stage + KG * 64 * SSTR;
#pragma unroll
  for (int q = 0; q < BM / 64; ++q) {
    // each K group stages its partial tile in a region of its own, all at
    // once; one pass then adds the regions in a fixed order (KG - 1 first,
    // 0 last) into region 0
    {
      float* reg = stage + kg * 64 * SSTR;
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        const int rb = wm * WM + i;  // 32-row block of the tile
        if (rb / 2 != q) continue;
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int rg = 0; rg < 16; ++rg) {
            const int r = 8 * (rg >> 2) + 4 * (lane >> 5) + (rg & 3);
            // (P16: the weights were stored scaled by 1 / wscale, a power of 2)
            reg[((rb & 1) * 32 + r) * SSTR + (wn * WN + j) * 32 + (lane & 31)] =
                P16 ? acc[i][j][rg] * a.wscale : acc[i][j][rg];
          }
      }
      __syncthreads();
      if constexpr (KG > 1) {
        constexpr int NQ4 = 64 * BN / 4;  // float4s of a pass
        for (int e = tid; e < NQ4; e += NT) {
          const int o = (e / (BN / 4)) * SSTR + 4 * (e % (BN / 4));
          float4 v = *reinterpret_cast<const float4*>(stage + (KG - 1) * 64 * SSTR + o);
#pragma unroll
          for (int g = KG - 2; g >= 0; --g) {
            const float4 w = *reinterpret_cast<const float4*>(stage + g * 64 * SSTR + o);
            v.x = v.x + w.x;
            v.y = v.y + w.y;
            v.z = v.z + w.z;
            v.w = v.w + w.w;
          }
          *reinterpret_cast<float4*>(stage + o) = v;
        }
        __syncthreads();
      }
    }
    if constexpr (EPI == GV_QKV) {
      qkv_tile_pass<BN, NT, P16>(a, stage, sinv, m0, n0, q, rows_fast, pos0);
      __syncthreads();
      continue;
    }
    // RELU2 writes planes only: items row-fastest, so 16 lanes store 256
    // consecutive bytes; RESID and STORE also touch row-major fp32: four
    // lanes per 128 bytes of a row
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int e = tid + k * NT;
      if (ITEMS % NT != 0 && e >= ITEMS) break;
      const int srow = EPI == GV_RELU2 ? e % 64 : e / (BN / 8);
      const int pc = 8 * (EPI == GV_RELU2 ? e / 64 : e % (BN / 8));
      const int ml = q * 64 + srow, m = m0 + ml, n = n0 + pc;
      const bool live = m < M;
      const float4 lo = *reinterpret_cast<const float4*>(stage + srow * SSTR + pc);
      const float4 hi = *reinterpret_cast<const float4*>(stage + srow * SSTR + pc + 4);
      float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      if (a.norm) {
        const float sc = sinv[ml];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] *= sc;
      }
      if (EPI == GV_RESID) {
        const float4 x0 = xres[q * EPT + k][0], x1 = xres[q * EPT + k][1];
        const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        float sq = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          v[i] = x[i] + v[i];
          sq += v[i] * v[i];
        }
        if (live) {
          f32x4_t* y = reinterpret_cast<f32x4_t*>(a.y + (int64_t)m * a.N + n);
          store_v<NT_RESID>(y, f32x4_t{v[0], v[1], v[2], v[3]});
          store_v<NT_RESID>(y + 1, f32x4_t{v[4], v[5], v[6], v[7]});
#pragma unroll
          for (int i = 0; i < 8; ++i) f16_guard<P16>(a, v[i]);
          put8<P16, NT_RESID>(v, a.ys + tile_at(m, n, a.N), a.ys_plane);
        }
        sqs[srow * SQS + pc / 8] = sq;
      } else if (EPI == GV_RELU2) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float t = v[i] < 0.f ? 0.f : v[i];
          v[i] = t * t;
          if (live) f16_guard<P16>(a, v[i]);
        }
        if (live) put8<P16, NT_RELU2>(v, a.ys + tile_at(m, n, a.N), a.ys_plane);
      } else if (live) {
        float4* y = reinterpret_cast<float4*>(a.y + (int64_t)m * a.N + n);
        y[0] = make_float4(v[0], v[1], v[2], v[3]);
        y[1] = make_float4(v[4], v[5], v[6], v[7]);
      }
    }
    __syncthreads();
    if constexpr (EPI == GV_RESID) {
      // four adjacent threads per row, each summing BN / 32 of its items in
      // column order, then a fixed butterfly
      constexpr int VPP = BN / 32;
      static_assert(NT >= 256 && VPP * 32 == BN, "row-sum split");
      if (tid < 256) {
        const int row = tid >> 2, part = tid & 3;
        float sum = 0.f;
#pragma unroll
        for (int v = 0; v < VPP; ++v) sum += sqs[row * SQS + part * VPP + v];
        sum += dpp_f<0xB1>(sum);  // lane ^ 1
        sum += dpp_f<0x4E>(sum);  // lane ^ 2
        if (part == 0 && m0 + q * 64 + row < M)
          a.ssq_out[(int64_t)(m0 + q * 64 + row) * (a.N / BN) + n0 / BN] = sum;
      }
      __syncthreads();
    }
  }
}

// ------------------------------------------------------------------ v2
// Wave tile (WM x 32) x (WN x 32), K slices of BK (32 or 64) per stage. The
// operand fragments of the next 16-deep step are read from LDS into a
// second register set while the MFMAs of the current one run (the last
// step of a slice runs after the next slice's barrier), so LDS latency hides
// behind MFMA work even at one wavefront per SIMD. The epilogue works
// straight from the accumulators, whose lane l holds column l % 32 of rows
// 8(r/4) + 4(l/32) + r%4, r = 0..15, of a 32x32 block: for the logits (STORE)
// 32 lanes write 32 consecutive columns of one row. For RELU2 the product is
// formed transposed (the same sums), so a lane holds 16 columns of one token
// row, and the two halves of a wavefront fill 16-byte chunks of the output
// tiles, 16 rows next to each other.
template <int WM, int WN>
struct Frag {
  bf16x8_t h[WM], l[WM], w[WN];
};

template <int BM, int WM, int WN, bool P16, int RT>
__device__ __forceinline__ void frag_load(Frag<WM, WN>& f, const uint8_t* stg, int kk, int wm,
                                          int wn, int lane) {
  constexpr int AP = P16 ? 1 : 2;
  const int c = 2 * kk + (lane >> 5);  // logical chunk of this half-wave
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int r = (wm * WM + i) * 32 + (lane & 31);
    f.h[i] = *(const bf16x8_t*)(stg + at<RT>(r, c));
    if constexpr (!P16) f.l[i] = *(const bf16x8_t*)(stg + at<RT>(BM + r, c));
  }
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int r = AP * BM + (wn * WN + j) * 32 + (lane & 31);
    f.w[j] = *(const bf16x8_t*)(stg + at<RT>(r, c));
  }
}

// TR: the transposed product (W rows down, token rows across).
template <int WM, int WN, bool P16, bool TR>
__device__ __forceinline__ void frag_mma(const Frag<WM, WN>& f, f32x16_t (&acc)[WM][WN]) {
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
      acc[i][j] = TR ? mma16<P16>(f.w[j], f.h[i], acc[i][j]) : mma16<P16>(f.h[i], f.w[j], acc[i][j]);
  if constexpr (!P16) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
        acc[i][j] = TR ? mma16<false>(f.w[j], f.l[i], acc[i][j])
                       : mma16<false>(f.l[i], f.w[j], acc[i][j]);
  }
}

template <int EPI, int NWM, int NWN, int WM, int WN, int NST, bool P16 = false, int BK = 32>
__global__ __launch_bounds__(64 * NWM * NWN) void k_gemm2(GemvArgs a) {
  static_assert(EPI == GV_RELU2 || EPI == GV_STORE, "register epilogues");
  constexpr bool TR = EPI == GV_RELU2;
  constexpr int BM = NWM * WM * 32, BN = NWN * WN * 32;
  constexpr int NW = NWM * NWN, NT = 64 * NW;
  constexpr int AP = P16 ? 1 : 2;
  constexpr int ROWS = AP * BM + BN, RT = ROWS / 16, GROUPS = RT * (BK / 32), GPW = GROUPS / NW;
  static_assert(GROUPS % NW == 0, "tile / wave grid mismatch");
  constexpr int STAGE_BYTES = GROUPS * 1024;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  __shared__ float sinv[BM];
  __shared__ int stgt[EPI == GV_STORE ? BM : 1];  // the rows' targets (a.nll_part)

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = wid / NWN, wn = wid % NWN;
  // XCD x runs a contiguous run of tiles in row-major order (see k_gemm)
  const int nbn = gridDim.x, ntile = gridDim.x * gridDim.y;
  int lin = blockIdx.x + nbn * blockIdx.y;
  if ((ntile & 7) == 0) lin = (lin & 7) * (ntile >> 3) + (lin >> 3);
  const int m0 = (lin / nbn) * BM, n0 = (lin % nbn) * BN;
  const int M = a.M, K = a.K;

  const uint16_t* src[GPW];
#pragma unroll
  for (int q = 0; q < GPW; ++q) {
    const int g = wid + NW * q, rt = g % RT, kt = g / RT;
    const uint16_t* base;
    if (rt < AP * (BM / 16)) {
      const int ar = rt < BM / 16 ? rt : rt - BM / 16;
      base = a.xs + (rt < BM / 16 ? 0 : a.xs_plane) +
             (int64_t)min((m0 >> 4) + ar, (M - 1) >> 4) * K * 16;
    } else {
      base = a.w + (int64_t)((n0 >> 4) + rt - AP * (BM / 16)) * K * 16;
    }
    src[q] = base + kt * 512 + lane * 8;
  }

  f32x16_t acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nk = K / BK, klast = K - BK;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_off(smem) + wid * 1024);
  auto fill = [&](int stg, int k0) {
#pragma unroll
    for (int q = 0; q < GPW; ++q) dma16(src[q] + k0 * 16, lds0 + stg * STAGE_BYTES + NW * q * 1024);
  };
#pragma unroll
  for (int si = 0; si < NST - 1; ++si) fill(si, min(si * BK, klast));
  Frag<WM, WN> f0, f1;
  for (int kt = 0; kt < nk; kt += NST) {
#pragma unroll
    for (int si = 0; si < NST; ++si) {
      if (kt + si < nk) {
        stage_sync<(NST - 2) * GPW>();
        fill((si + NST - 1) % NST, min((kt + si + NST - 1) * BK, klast));
        const uint8_t* stg = smem + si * STAGE_BYTES;
        frag_load<BM, WM, WN, P16, RT>(f0, stg, 0, wm, wn, lane);
        if (kt + si > 0) frag_mma<WM, WN, P16, TR>(f1, acc);  // last k-step of the previous slice
        frag_load<BM, WM, WN, P16, RT>(f1, stg, 1, wm, wn, lane);
        frag_mma<WM, WN, P16, TR>(f0, acc);
#pragma unroll
        for (int kk = 2; kk < BK / 16; kk += 2) {
          frag_load<BM, WM, WN, P16, RT>(f0, stg, kk, wm, wn, lane);
          frag_mma<WM, WN, P16, TR>(f1, acc);
          frag_load<BM, WM, WN, P16, RT>(f1, stg, kk + 1, wm, wn, lane);
          frag_mma<WM, WN, P16, TR>(f0, acc);
        }
      }
    }
  }
  frag_mma<WM, WN, P16, TR>(f1, acc);
  wait_vmcnt<0>();

  if (a.norm) {
    for (int r = tid; r < BM; r += NT) {
      float ssum = 0.f;
      if (m0 + r < M)
        for (int t = 0; t < a.ssq_n; ++t) ssum += a.ssq_in[(int64_t)(m0 + r) * a.ssq_n + t];
      sinv[r] = 1.0f / sqrtf(ssum / (float)K + a.eps);
    }
  }
  if (EPI == GV_STORE && a.nll_part)
    for (int r = tid; r < BM; r += NT) stgt[r] = m0 + r < M ? a.tgt[m0 + r] : -1;
  __syncthreads();

  const int half = lane >> 5, cl = lane & 31;
  if constexpr (TR) {
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int ml = (wm * WM + i) * 32 + cl, m = m0 + ml;
      if (m >= M) continue;
      const float sc = (a.norm ? sinv[ml] : 1.f) * (P16 ? a.wscale : 1.f);  // (wscale: a power of 2)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const int n = n0 + (wn * WN + j) * 32 + 8 * rq + 4 * half;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float u = acc[i][j][4 * rq + e] * sc, t = u < 0.f ? 0.f : u;
            v[e] = t * t;
            f16_guard<P16>(a, v[e]);
          }
          put4<P16>(v, a.ys + tile_at(m, n, a.N), a.ys_plane);
        }
    }
    return;
  }
  // The cross-entropy's part (a.nll_part): per row and NLL_GROUP_COLS columns
  // (this wavefront's), the maximum and the sum of exp(v - max) (the hardware
  // exp2 of (v - max) log2 e: its relative error, a few ulp, is far below the
  // tolerance of the nll), and the target's logit from whichever lane holds
  // it. The values are the logits stored, bit for bit; a.y null: not stored.
  // Row 8 (r / 4) + 4 half + r % 4 of a 32-row block is kept by lane r of the
  // half, so a block's partials leave in one store.
  constexpr bool CAN_NLL = EPI == GV_STORE && WN * 32 == NLL_GROUP_COLS;
  const bool nll = CAN_NLL && a.nll_part;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int rb = (wm * WM + i) * 32 + 4 * half;  // tile row of r = 0
    float pm = 0.f, ps = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int rl = rb + 8 * (r >> 2) + (r & 3), m = m0 + rl;
      const float inv = a.norm ? sinv[rl] : 1.f;
      float v[WN];
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        v[j] = (P16 ? acc[i][j][r] * a.wscale : acc[i][j][r]) * inv;
        if (m < M && (!CAN_NLL || a.y))  // logits: read once, later
          __builtin_nontemporal_store(v[j], a.y + (int64_t)m * a.N + n0 + (wn * WN + j) * 32 + cl);
      }
      if constexpr (CAN_NLL) {
        if (nll) {
          const int t = stgt[rl] - n0 - wn * WN * 32 - cl;  // (-1 for rows past M)
          float mx = v[0], e = 0.f;
#pragma unroll
          for (int j = 0; j < WN; ++j) {
            if (t == 32 * j) a.tlogit[m] = v[j];
            mx = fmaxf(mx, v[j]);
          }
          mx = half_max_swap(mx);
#pragma unroll
          for (int j = 0; j < WN; ++j) e += __expf(v[j] - mx);
          e = half_sum_swap(e);
          pm = cl == r ? mx : pm;
          ps = cl == r ? e : ps;
        }
      }
    }
    if constexpr (CAN_NLL) {
      const int m = m0 + rb + 8 * (cl >> 2) + (cl & 3);
      if (nll && cl < 16 && m < M)
        *reinterpret_cast<float2*>(a.nll_part + ((int64_t)m * (a.N / NLL_GROUP_COLS) +
                                                 n0 / NLL_GROUP_COLS + wn) * 2) = make_float2(pm, ps);
    }
  }
}

template <int EPI, int NWM, int NWN, int WM, int WN, int NST, bool P16, int BK = 32>
void launch_cfg2(hipStream_t s, const GemvArgs& a) {
  constexpr int BM = NWM * WM * 32, BN = NWN * WN * 32;
  constexpr size_t lds = (size_t)NST * ((P16 ? 1 : 2) * BM + BN) * 2 * BK;
  static_assert(lds + BM * sizeof(float) <= 160 * 1024, "tile exceeds the LDS");
  static std::atomic<uint64_t> attr{0};
  raise_lds_once((const void*)k_gemm2<EPI, NWM, NWN, WM, WN, NST, P16, BK>, lds, &attr);
  const dim3 g(a.N / BN, (unsigned)((a.M + BM - 1) / BM));
  FG_LAUNCH((k_gemm2<EPI, NWM, NWN, WM, WN, NST, P16, BK>), g, dim3(64 * NWM * NWN), lds, s, a);
}

template <int EPI, int BM, int BN, int NWM, int NWN, int BK, int NST, int KG, bool P16>
void launch_cfg(hipStream_t s, const GemvArgs& a, const int32_t* d_pos) {
  constexpr size_t pipe = (size_t)NST * ((P16 ? 1 : 2) * BM + BN) * 2 * BK;
  constexpr size_t epi =
      (size_t)KG * 64 * (BN + 4) * 4 + (EPI == GV_RESID ? (size_t)64 * (BN / 8 + 1) * 4 : 0);
  constexpr size_t lds = pipe > epi ? pipe : epi;
  // gfx950: 160 KB of LDS per workgroup, the row scales (BM floats) included
  static_assert(lds + BM * sizeof(float) <= 160 * 1024, "tile exceeds the LDS");
  static std::atomic<uint64_t> attr{0};
  raise_lds_once((const void*)k_gemm<EPI, BM, BN, NWM, NWN, BK, NST, KG, P16>, lds, &attr);
  const dim3 g(a.N / BN, (unsigned)((a.M + BM - 1) / BM));
  FG_LAUNCH((k_gemm<EPI, BM, BN, NWM, NWN, BK, NST, KG, P16>), g, dim3(64 * NWM * NWN * KG),
                     lds, s, a, d_pos);
}

// 128 wide while that still leaves half the CUs a block (the wider tile
// reads the A panel half as often), else 64 wide
int tile_n(int64_t M, int N) {
  const int64_t mt64 = (M + 63) / 64;
  return (N % 128 == 0 && mt64 * (N / 128) >= 128) ? 128 : 64;
}

// The residual GEMMs whose 64x64 tiles fit the CUs in one round: no CU has
// more to do, and none would idle for a wider tile (M = 1280, N = 768, 240
// tiles against 160 of 64x96: fp16 proj2 18.4 -> 13.6 us, split 24.9 -> 19.5).
bool resid_64(int64_t M, int N) {
  return N % 64 == 0 && (M + 63) / 64 * (N / 64) <= cu_count();
}

// The residual GEMMs whose 128x128 tiles give half of the CUs or more one each
// (and 64x96, 64x128 or 64x160 ones do not fit one round): M = 3072, N = 768
// (144 tiles), against 64x128 ones: proj2 fp16 32.4 -> 27.9 us, split 58.5 ->
// 45.5; M = 3072, N = 1280 (240) 59.3 -> 51.5, 103.7 -> 86.3; but M = 1554, N =
// 1280 (130) 69.3 split, where one round of 64x128 tiles (200 at M = 1280)
// takes 48.0.
bool resid_128(int64_t M, int N) {
  return N % 128 == 0 && 2 * ((M + 127) / 128 * (N / 128)) >= cu_count() &&
         (M + 63) / 64 * (N / 128) > cu_count();
}

// lm_head on 256x256 tiles: past half a round of them over the CUs (three
// quarters with split operands: at 160 tiles fp16 37.4 -> 29.9 us, split 40.9
// -> 42.3 and more).
bool store_256(int64_t M, int N, bool f16) {
  const int64_t t = (M + 255) / 256 * (N / 256), ncu = cu_count();
  return N % 256 == 0 && 4 * t > (f16 ? 2 : 3) * ncu;
}

// The residual GEMMs (proj, proj2) at prefill sizes, where 64x128 tiles
// leave CUs idle and 64x96 tiles give more than half of them one each
// (M = 2048, N = 768: 256 tiles): 64x96 tiles with K split over 4
// wavefront groups, two wavefronts per SIMD (measured 2-4 us a launch
// faster than 64x128 tiles at one wavefront per SIMD).
bool resid_k4(int64_t M, int N, int K) {
  const int64_t mt64 = (M + 63) / 64, ncu = cu_count(), t96 = mt64 * (N / 96);
  return K % 64 == 0 && N % 96 == 0 && mt64 * (N / 128) < ncu && t96 <= ncu && 2 * t96 > ncu;
}

// The residual GEMMs where 64x128 tiles spill into a second round over the
// CUs and 64x160 tiles fill one (the depth-20 model's d_model 1280 at 2047
// rows: 320 tiles of 64x128, 256 of 64x160): K split over 2 wavefront
// groups of two (the staged tiles of four groups would not fit the LDS).
bool resid_160(int64_t M, int N, int K) {
  const int64_t mt64 = (M + 63) / 64, ncu = cu_count(), t160 = mt64 * (N / 160);
  return K % 64 == 0 && N % 160 == 0 && mt64 * (N / 128) > ncu && t160 <= ncu &&
         2 * t160 > ncu;
}

// Tile choice. The LDS-staged epilogue (k_gemm) serves QKV and RESID at every
// size, whose outputs are scattered or need per-row reductions, the 128x192
// tiles of RELU2, and both plain stores below 256 tiles of 128x128; the register
// epilogue (k_gemm2) serves the larger RELU2 and lm_head GEMMs: 128x128 tiles,
// RELU2 on 128x256 ones (wave 64x128) from 3 blocks per CU on, lm_head on
// 256x256 or (8 wavefronts) 128x256 ones by the rules below, and either on
// 256x256 past 4096 rows in fp16.

template <int EPI, bool P16>
void launch_tile_p(hipStream_t s, const GemvArgs& a, const int32_t* d_pos) {
  if constexpr (P16 && (EPI == GV_RELU2 || EPI == GV_STORE)) {
    // single-term fc and lm_head over more than 4096 rows: 256x256 tiles (8
    // wavefronts of 128x64; one fp16 A plane leaves room for them), 4 % of
    // the GEMM time faster than 128x256 over 8 x 2048 rows in the layer stack;
    // two 64-wide K slices (128 KB) rather than three 32-wide ones, half the
    // barriers per K: 0.8 % of the 8 x 2048 eval forward (identical bits; at
    // 2048 rows the 128x256 tiles are 1.5 % slower with them)
    if (a.M > 4096 && a.N % 256 == 0) {
      launch_cfg2<EPI, 2, 4, 4, 2, 2, P16, 64>(s, a);
      return;
    }
  }
  if constexpr (EPI == GV_STORE) {
    // lm_head: 256x256 tiles (also the ones whose epilogue writes the
    // cross-entropy's partials); in front of them 128x256 where those cover
    // most of the CUs once. us, before (128x256 in 4 wavefronts, 128x128) ->
    // after, d_model 768, fp16 / split: M = 2048 51.0 -> 37.9 / 62.2 -> 52.7,
    // 4096 98 -> 72 / 122 -> 101, 600 20.9 -> 16.0 / 25.6 -> 22.0, 800 25.7 ->
    // 23.3 / 28.5 -> 26.6
    if (store_256(a.M, a.N, P16)) {
      launch_cfg2<EPI, 2, 4, 4, 2, 2, P16>(s, a);
      return;
    }
    const int64_t t256 = (a.M + 127) / 128 * (a.N / 256), ncu = cu_count();
    if (a.N % 256 == 0 && 8 * t256 >= 5 * ncu && t256 <= ncu) {
      launch_cfg2<EPI, 2, 4, 2, 2, 3, P16>(s, a);
      return;
    }
  }
  const int64_t mt128 = (a.M + 127) / 128;
  // fc at prefill sizes: where 128x128 tiles spill into a second, mostly
  // empty round over the CUs, 128x192 tiles fit in one (QKV stays on
  // 128x128: its epilogue costs more per column in the wider tile)
  if constexpr (EPI == GV_RELU2) {
    const int64_t ncu = cu_count();
    if (a.N % 192 == 0 && a.K % 64 == 0 && mt128 * (a.N / 128) > ncu &&
        mt128 * (a.N / 192) <= ncu) {
      launch_cfg<EPI, 128, 192, 4, 2, 64, 2, 1, P16>(s, a, d_pos);
      return;
    }
  }
  const bool big = a.N % 128 == 0 && mt128 * (a.N / 128) >= 256;
  if constexpr (EPI == GV_RELU2 || EPI == GV_STORE) {
    if (EPI == GV_RELU2 && a.N % 256 == 0 && mt128 * (a.N / 256) >= 768) {
      launch_cfg2<EPI, 2, 2, 2, 4, 2, P16>(s, a);
      return;
    }
    if (big) {
      launch_cfg2<EPI, 4, 2, 1, 2, 3, P16>(s, a);
      return;
    }
  }
  if constexpr (EPI == GV_RESID) {
    if (resid_64(a.M, a.N)) {
      // K over 4 wavefront groups (two wavefronts a SIMD) except where the
      // split operands and a short K keep one group busy. us: fp16 M = 450
      // proj2 (K = 3072) 15.6 -> 12.3, 1024 16.2 -> 12.8, M = 300 at K = 5120
      // 22.9 -> 17.0, proj (K = 768) 6.5 -> 6.1; split M = 1024 proj2 18.9 ->
      // 18.8, proj 7.9 on one group, more on four
      if (a.K % 64 == 0 && (P16 || a.K >= 2048))
        launch_cfg<EPI, 64, 64, 2, 1, 64, 4, 4, P16>(s, a, d_pos);
      else
        launch_cfg<EPI, 64, 64, 2, 2, 32, 4, 1, P16>(s, a, d_pos);
      return;
    }
    if (resid_k4(a.M, a.N, a.K)) {
      launch_cfg<EPI, 64, 96, 2, 1, 64, 3, 4, P16>(s, a, d_pos);
      return;
    }
    if (resid_160(a.M, a.N, a.K)) {
      launch_cfg<EPI, 64, 160, 2, 1, 64, 3, 2, P16>(s, a, d_pos);
      return;
    }
    if (resid_128(a.M, a.N) && !big) {
      launch_cfg<EPI, 128, 128, 4, 2, 32, 3, 1, P16>(s, a, d_pos);
      return;
    }
  }
  const int bn = tile_n(a.M, a.N);
  if constexpr (EPI == GV_QKV) {
    // 128x128 tiles from where 64x128 ones would need a second round (the
    // depth-20 model at 2047 rows: 224 tiles against 448), but for the second
    // case here
    const int64_t ncu = cu_count(), t128 = mt128 * (a.N / 128);
    const int64_t t64 = (int64_t)((a.M + 63) / 64) * (a.N / 128);
    // 64x64 tiles while 64x128 ones would leave CUs without one: us, fp16 /
    // split: M = 450, N = 2304 12.4 -> 9.9 / 14.0 -> 12.0, 800 11.3 -> 9.8 /
    // 14.2 -> 13.2
    if (bn == 128 && t64 <= ncu) {
      launch_cfg<EPI, 64, 64, 2, 2, 32, 4, 1, P16>(s, a, d_pos);
      return;
    }
    // 64x128 tiles where 128x128 ones fill one or two rounds over the CUs and
    // less than half of the next: M = 1800, N = 2304 (270) 20.4 -> 19.1 / 29.6
    // -> 27.0, 2048 (288) 19.8 -> 19.9 / 28.6 -> 26.2, 4096 (576) 32.5 -> 31.2 /
    // 44.1 -> 42.0; M = 3072, N = 1792 (336) 29.4 -> 27.6 / 43.6 -> 38.5
    if (bn == 128 && a.K % 64 == 0 && t128 > ncu && t128 < 3 * ncu && 2 * (t128 % ncu) < ncu) {
      if constexpr (P16) launch_cfg<EPI, 64, 128, 2, 2, 64, 2, 1, P16>(s, a, d_pos);
      else launch_cfg<EPI, 64, 128, 2, 2, 32, 3, 1, P16>(s, a, d_pos);
      return;
    }
    if (bn == 128 && !big) {
      launch_cfg<EPI, 128, 128, 4, 2, 32, 3, 1, P16>(s, a, d_pos);
      return;
    }
  }
  if (P16 && bn == 128 && big && EPI != GV_STORE && a.M > 1024 && a.K % 64 == 0)
    // single-term QKV and residual GEMMs that fill the chip with 128x128
    // tiles: 64-wide K slices, two stages (64 KB with one fp16 A plane):
    // 1-3 % of the GEMM time faster than 32-wide ones over 8 x 2048 rows,
    // and the depth-12 forward 0.9 % (1 x 2048) to 1.2 % (2 x 2048) faster
    launch_cfg<EPI, 128, 128, 4, 2, 64, 2, 1, P16>(s, a, d_pos);
  else if (bn == 128 && big)
    launch_cfg<EPI, 128, 128, 4, 2, 32, 3, 1, P16>(s, a, d_pos);  // 72 KB: two blocks per CU
  else if (bn == 128 && EPI == GV_RESID && a.K % 64 == 0)
    // the residual GEMMs (proj, proj2) inside the layer stack: 64-wide slices
    // (half the stage hand-overs) measured ~4 us a launch faster than 32-wide
    // ones at any depth
    launch_cfg<EPI, 64, 128, 2, 2, 64, 3, 1, P16>(s, a, d_pos);
  else if (bn == 128) {
    if constexpr (EPI != GV_QKV) launch_cfg<EPI, 64, 128, 2, 2, 32, 4, 1, P16>(s, a, d_pos);
  } else
    launch_cfg<EPI, 64, 64, 2, 2, 32, 4, 1, P16>(s, a, d_pos);
}

template <int EPI>
void launch_tile(hipStream_t s, const GemvArgs& a, const int32_t* d_pos) {
  if (gemm_rows_tile(a.M, a.N).tm > 0) {  // few token rows
    launch_gemm_rows(s, (GemvEpi)EPI, a, d_pos);
    return;
  }
  if (a.f16)
    launch_tile_p<EPI, true>(s, a, d_pos);
  else
    launch_tile_p<EPI, false>(s, a, d_pos);
}

}  // namespace

// Compute units of the current device (tile counts are weighed against it).
int cu_count() {
  static std::atomic<int> n[64];  // 0: not looked up yet (handles on several threads)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = n[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        v <= 0)
      v = 256;
    n[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// lm_head writes the log-sum-exp partials where it runs on 256x256 tiles, up to
// 4096 rows (a row's 64 columns of a wavefront meet by DPP and one row swap),
// and then stores no logits where none are asked for. Past that its reductions,
// 11 us a round of tiles, cost more than a pass over stored logits: 16384 rows
// 387 us against 271 + 94. Whole pass of 2048 rows, logits and cross-entropy,
// fp16: 1254 us with a pass over the stored logits, 1245 so.
bool gemm_store_nll(int64_t M, int N, bool f16) {
  return M <= GEMM_NLL_ROWS && gemm_rows_tile(M, N).tm == 0 && store_256(M, N, f16);
}

// RESID: one sum-of-squares partial per row and N tile.
int gemm_ssq_parts(int64_t M, int N, int K) {
  if (const RowsTile t = gemm_rows_tile(M, N); t.tm > 0) return N / (16 * t.tn);
  if (resid_64(M, N)) return N / 64;
  if (resid_k4(M, N, K)) return N / 96;
  if (resid_160(M, N, K)) return N / 160;
  if (resid_128(M, N)) return N / 128;
  return N / tile_n(M, N);
}

int64_t gemm_ssq_floats(int64_t M, int N) {
  return std::max(std::min(M, ROWS_MAX_M) * (N / 16), M * (N / 64));
}

void launch_gemm_pos(hipStream_t s, GemvEpi epi, const GemvArgs& a, const int32_t* d_pos) {
  switch (epi) {
    case GV_QKV: launch_tile<GV_QKV>(s, a, d_pos); break;
    case GV_RESID: launch_tile<GV_RESID>(s, a, d_pos); break;
    case GV_RELU2: launch_tile<GV_RELU2>(s, a, d_pos); break;
    default: launch_tile<GV_STORE>(s, a, d_pos); break;
  }
}

}  // namespace fgpt
