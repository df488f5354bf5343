// kern_sample.h -- sample_next of src/lib/sample.f90:153-233 for one row of
// logits: what both device forms share (the generator, the sort keys, the
// penalties), and the form that the persistent decode runs between two of its
// steps (sample_wg).
#pragma once
#include <float.h>

#include "fgpt_internal.h"
#include "kern_common.h"

namespace fgpt {
namespace {

// xorshift64* of rand_u01: the state advances, the top 24 bits of
// state * 2685821657736338717 give u in [0, 1)
__device__ __forceinline__ float rand_u01(int64_t* st) {
  uint64_t x = (uint64_t)*st;
  if (x == 0) x = 2685821657736338717ull;
  x ^= x << 13;
  x ^= x >> 7;
  x ^= x << 17;
  *st = (int64_t)x;
  const uint64_t y = x * 2685821657736338717ull;
  return (float)((y >> 40) & 0xFFFFFFull) / 16777216.0f;
}

// Sort keys: the probability's bits (p >= 0, so they order as p does) above,
// 0x7fffffff - id below: descending key order is descending probability
// with ties in ascending id; key 0 (padding past V) sorts last.
__device__ __forceinline__ uint64_t prob_key(float p, int id) {
  return ((uint64_t)__float_as_uint(p) << 32) | (uint32_t)(0x7fffffff - id);
}

// The row's penalties, n-gram ban and byte mask, in the reference's order:
// presence and frequency over the whole history or its last pwin ids (:33-51,
// :77-104), the repetition penalty (:56-71), the no-repeat n-gram ban
// (:109-130), the byte-level ids (:141-151). X is how the caller's threads
// split an index range (each), meet (sync), read an id of the history (id) and
// count it from an index on (count, then n_of).
template <class X>
__device__ __forceinline__ void penalise(X& x, float* pr, int V, int ngen, const SampleCfg& c) {
#pragma clang fp contract(off)
  const int lo = c.pwin > 0 && ngen > c.pwin ? ngen - c.pwin : 0;
  if ((c.pres != 0.f || c.freq != 0.f) && ngen > 0) {  // l - pres - freq * count
    x.count(lo);
    x.each(0, V, [&](int i) {
#pragma clang fp contract(off)
      const int n = x.n_of(i);
      if (n > 0) pr[i] = (pr[i] - c.pres) - c.freq * (float)n;
    });
    x.sync();
  }
  if (c.pwin > 0 && ngen > 0 && c.plen != 0.f && ngen < c.pwin) {
    if (threadIdx.x == 0) pr[0] = pr[0] - (c.plen * (float)(c.pwin - ngen)) / (float)c.pwin;
    x.sync();
  }
  if (c.rep > 1.f && ngen > 0) {  // over the whole history: l / theta
    x.count(0);
    x.each(0, V, [&](int i) {
      if (x.n_of(i) > 0) pr[i] = pr[i] / c.rep;
    });
    x.sync();
  }
  const int nn = c.nblock;
  if (nn >= 2 && ngen >= nn) {  // ids that would complete an n-gram of the history
    x.each(0, ngen - nn + 1, [&](int s) {
      int k = 0;
      while (k < nn - 1 && x.id(s + k) == x.id(ngen - nn + 1 + k)) ++k;
      if (k == nn - 1) {
        const int t = x.id(s + nn - 1);
        if (t >= 0 && t < V) pr[t] = -FLT_MAX;
      }
    });
    x.sync();
  }
  if (c.byte_space) {
    x.each(0, V, [&](int i) {
      if (!(i < 128 || (i >= 256 && i < 512))) pr[i] = -FLT_MAX;
    });
    x.sync();
  }
}

// How 256 of a workgroup's threads (comp; the others only keep the barriers) go
// through penalise().
template <int V>
struct WalkWG {
  uint32_t* cnt;  // [V / 2]: 16-bit counts, two a word (histories are below 2^16)
  const int32_t* gen;
  int ngen;
  bool comp;
  int counted = -1;  // history start that cnt holds
  template <class F>
  __device__ __forceinline__ void each(int lo, int hi, F&& f) {
    if (comp)
      for (int i = lo + (int)threadIdx.x; i < hi; i += 256) f(i);
  }
  __device__ __forceinline__ void sync() { lds_barrier(); }
  // (the history is this workgroup's own stores of earlier steps)
  __device__ __forceinline__ int id(int j) {
    return __hip_atomic_load(gen + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ void count(int lo) {
    if (counted == lo) return;
    counted = lo;
    each(0, V / 2, [&](int i) { cnt[i] = 0; });
    lds_barrier();
    each(lo, ngen, [&](int j) {
      const int g = id(j);
      if (g >= 0 && g < V) atomicAdd(&cnt[g >> 1], 1u << (16 * (g & 1)));
    });
    lds_barrier();
  }
  __device__ __forceinline__ int n_of(int i) {
    return (int)((cnt[i >> 1] >> (16 * (i & 1))) & 0xFFFFu);
  }
};

// The sampling of one row by 256 of a workgroup's threads (comp; the others
// only keep the barriers), V a power of two, from pr[V] in LDS, which is
// overwritten; aux: sample_wg_aux(V) bytes of LDS. The draw is sample_row's
// (kern_sample.hip) bit for bit: the same sums in the same order (SVT threads'
// strided partials; 8 entries, then 64 of their totals, then the rest).
//
// What bounds it is its chain of block-wide steps, so the sort, by far the
// longest, is cut down to what the draw can reach: the ids of probability at
// least 2^-k of the largest, for the first k whose mass passes topp (by 1e-3,
// far more than the sums' rounding). The cut is in probabilities, so no run of
// equal ones straddles it, and the kept prefix of the order, its cumulative
// sums included, is that of the whole row. Where no such cut keeps V / 8 ids or
// fewer (flat rows, topp near 1 or above) the row would have to be sorted whole,
// 240 us on 256 threads against k_sample_step's 52 on 1024: SAMPLE_WHOLE is
// returned instead, nothing drawn, and the loop ends so that the caller goes on
// with that kernel.
// A drawn id of the depth-12 model after 120 positions: 222 us with a launch
// of the step and one of k_sample_step (52 us) an id, 163 in the loop, of
// which a step with its argmax takes 137.
constexpr int SVT = 1024;  // threads that sample_row's sums are split over
constexpr int64_t sample_wg_aux(int V) { return 2 * V + 4 * SVT + 256; }
constexpr int SAMPLE_WHOLE = 1 << 30;  // (no id: vocabularies are far smaller)

template <int V>
__device__ int sample_wg(float* pr, uint8_t* aux, const int32_t* gen, int ngen, const SampleCfg& c,
                         int64_t* state, bool comp) {
#pragma clang fp contract(off)
  constexpr int NT = 256, PER = V / SVT, MAXC = V / 8, NK = 6;
  static_assert(V >= SVT && (V & (V - 1)) == 0 && 8 * MAXC <= 2 * V, "V a power of two");
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  uint64_t* keys = (uint64_t*)aux;      // [MAXC]
  float* tot = (float*)(aux + 2 * V);   // [SVT]
  float* red = tot + SVT;               // [16]
  int* ri = (int*)(red + 16);           // [16]
  float* mred = (float*)(ri + 16);      // [4] and a broadcast
  WalkWG<V> walk{(uint32_t*)aux, gen, ngen, comp};
  penalise(walk, pr, V, ngen, c);
  if (c.temp <= 0.f) {  // the first maximum, no draw
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    if (comp) {
      for (int i = tid; i < V; i += NT)
        if (pr[i] > bv) {
          bv = pr[i];
          bi = i;
        }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const float v2 = __shfl_xor(bv, o, 64);
        const int i2 = __shfl_xor(bi, o, 64);
        if (v2 > bv || (v2 == bv && i2 < bi)) {
          bv = v2;
          bi = i2;
        }
      }
      if (lane == 0) {
        red[wv] = bv;
        ri[wv] = bi;
      }
    }
    lds_barrier();
    bv = red[0];
    bi = ri[0];
    for (int k = 1; k < 4; ++k)
      if (red[k] > bv || (red[k] == bv && ri[k] < bi)) {
        bv = red[k];
        bi = ri[k];
      }
    return bi == 0x7fffffff ? 0 : bi;
  }

  // softmax at the temperature
  const float t = c.temp < 1.0e-6f ? 1.0e-6f : c.temp;
  if (comp) {
    float m = -INFINITY;
    for (int i = tid; i < V; i += NT) m = fmaxf(m, pr[i]);
    m = wave_max(m);
    if (lane == 0) mred[wv] = m;
  }
  lds_barrier();
  const float m = fmaxf(fmaxf(mred[0], mred[1]), fmaxf(mred[2], mred[3]));
  if (comp) {
#pragma unroll 1
    for (int k = 0; k < SVT / NT; ++k) {  // sample_row's thread tid + 256 k
      float part = 0.f;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int i = tid + NT * k + SVT * j;
        const float e = expf((pr[i] - m) / t);
        pr[i] = e;
        part += e;
      }
      part = wave_sum(part);
      if (lane == 0) red[4 * k + wv] = part;
    }
  }
  if (tid == 0) ri[15] = 0;
  lds_barrier();
  float s = 0.f;
  for (int k = 0; k < SVT / 64; ++k) s += red[k];

  // probabilities, and the mass and count at or above each cut
  const float pmax = 1.0f / s;  // (the largest e is exp(0))
  if (comp) {
    float ms[NK];
    int ns[NK];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      ms[k] = 0.f;
      ns[k] = 0;
    }
#pragma unroll 2
    for (int i = tid; i < V; i += NT) {
      const float p = pr[i] / s;
      pr[i] = p;
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const bool in = p >= pmax * (1.f / (float)(8 << (2 * k)));
        ms[k] += in ? p : 0.f;
        ns[k] += in ? 1 : 0;
      }
    }
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const float a = wave_sum(ms[k]), n = wave_sum((float)ns[k]);
      if (lane == 0) {
        tot[8 * wv + k] = a;
        tot[32 + 8 * wv + k] = n;
      }
    }
  }
  lds_barrier();
  float tau = 0.f;
  int nc = 0;  // ids kept
#pragma unroll
  for (int k = NK - 1; k >= 0; --k) {
    const float mass = (tot[k] + tot[8 + k]) + (tot[16 + k] + tot[24 + k]);
    const float n = (tot[32 + k] + tot[40 + k]) + (tot[48 + k] + tot[56 + k]);
    if (mass >= c.topp + 1e-3f && n <= (float)MAXC) {
      tau = pmax * (1.f / (float)(8 << (2 * k)));
      nc = (int)n;
    }
  }
  if (nc == 0) {
    lds_barrier();  // (pr and aux are free again)
    return SAMPLE_WHOLE;
  }
  int n2 = 64;
  while (n2 < nc) n2 <<= 1;
  if (comp) {
    for (int i = tid; i < V; i += NT)
      if (pr[i] >= tau) keys[atomicAdd(&ri[15], 1)] = prob_key(pr[i], i);
    for (int i = nc + tid; i < n2; i += NT) keys[i] = 0ull;
  }
  lds_barrier();
  // bitonic, descending; steps of j < 128 stay within the 128 keys that a
  // wavefront's 64 pairs span
  for (int k = 2; k <= n2; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (comp)
        for (int q = tid; q < n2 / 2; q += NT) {
          const int i = 2 * q - (q & (j - 1));
          const uint64_t x = keys[i], y = keys[i + j];
          if ((x < y) == ((i & k) == 0)) {
            keys[i] = y;
            keys[i + j] = x;
          }
        }
      if (j >= 128 || (j == 1 && k >= 128))
        lds_barrier();
      else
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  lds_barrier();
  // cumulative sums, into pr: PER entries a (sample_row) thread, 64 threads'
  // totals, then the groups of 64
  const int ngrp = (nc + 64 * PER - 1) / (64 * PER), nv = comp ? 64 * ngrp : 0;
#pragma unroll 1
  for (int v = tid; v < nv; v += NT) {
    float run = 0.f;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int i = v * PER + q;
      run += i < nc ? __uint_as_float((uint32_t)(keys[i] >> 32)) : 0.f;
      pr[i] = run;
    }
    tot[v] = run;
  }
  lds_barrier();
  if (tid < ngrp) {
    float a = 0.f;
#pragma unroll 1
    for (int q0 = 0; q0 < 64; q0 += 16) {
      float w[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) w[q] = tot[tid * 64 + q0 + q];
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        a += w[q];
        tot[tid * 64 + q0 + q] = a;
      }
    }
    red[tid] = a;
  }
  lds_barrier();
  int first = 0x7fffffff;
#pragma unroll 1
  for (int v = tid; v < nv; v += NT) {
    float base = 0.f;
    for (int g = 0; g < (v >> 6); ++g) base += red[g];
    const float off = base + ((v & 63) ? tot[v - 1] : 0.f);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int i = v * PER + q;
      const float a = pr[i] + off;
      pr[i] = a;
      if (a >= c.topp && i < first) first = i;
    }
  }
  auto block_min = [&](int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    if (comp && lane == 0) ri[wv] = v;
    lds_barrier();
    const int r = min(min(ri[0], ri[1]), min(ri[2], ri[3]));
    lds_barrier();
    return r;
  };
  int cut = V;
  first = block_min(first);
  if (c.topp < 1.f) cut = first < V ? first + 1 : V;
  if (tid == 0) mred[4] = rand_u01(state) * pr[cut - 1];
  lds_barrier();
  const float u = mred[4];
  int hit = 0x7fffffff;
  if (comp)
    for (int i = tid; i < min(cut, nc); i += NT)
      if (pr[i] >= u && i < hit) hit = i;
  hit = block_min(hit);
  hit = hit < cut ? hit : cut - 1;
  const int id = 0x7fffffff - (int)(uint32_t)keys[hit];
  lds_barrier();  // (pr and aux are free again)
  return id;
}

}  // namespace
}  // namespace fgpt
