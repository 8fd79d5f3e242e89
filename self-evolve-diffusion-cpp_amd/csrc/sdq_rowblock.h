// Rows held in registers across their serial sums: one workgroup of eight
// waves per 14 rows. Seven waves hold two whole rows each (lane l: 4 columns
// at 256 i + 4 l of chunk i), so a row norm reads its rows once and writes its
// result once. The sums keep the reference's column order (bit-exact, see
// sdq_rowsum.h): chunk by chunk those waves put their terms into a ring in
// LDS, and the eighth, its lane l on row l % 14, runs the dependent adds of all
// rows (a wave of its own: its operand tiles and the rows would not fit
// one wave's registers at two workgroups per CU; five-wave workgroups of eight
// rows, which place two waves on one SIMD, ran one or two per CU).
//
// What bounds it: HBM for many rows (two workgroups per CU overlap their
// loads, chains and stores), the chain of dependent adds for few (a
// 3072-column chain is ~7 us). It replaces, for rows of up to 3072 columns, a
// statistics kernel that reads the rows once per sum and an apply kernel. us
// before and after, 3072 columns: rmsnorm + RoPE of q and k at 27280 rows 531,
// 280 (4.8 TB/s), at 768 rows 26, 18.3; layernorm at 27280 rows 354, 180, at
// 157 rows 29, 22.5; norm + modulation + quantizer at 27280 rows 196, 150-170,
// at 4099 rows 60, 41, at 768 rows 35, 26.7.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "sdq_rowsum.h"

namespace sdq {
namespace rowblock {

constexpr int kRows = 14;      // rows per workgroup
constexpr int kWaves = 7;      // that hold rows
constexpr int kThreads = 64 * (kWaves + 1);
constexpr int kChunk = 256;    // columns per chunk
constexpr int kMaxChunks = 12;
constexpr int64_t kMaxCols = kMaxChunks * kChunk;
// Rows of one launch (of 32-row fragments); more run as several. A grid of 2^32
// threads or more wraps without an error.
constexpr int64_t kMaxRows = ((int64_t(1) << 32) - 1) / kThreads * kRows / 32 * 32;
// Many narrow rows stay with the two-kernel form: a workgroup adds 512 columns
// whatever the row's width. us, two kernels / one pass, 200000 rows: layernorm
// of 4 columns 62 / 97, of 20 80 / 99, of 28 102 / 100; rmsnorm + RoPE of 4
// columns 35 / 75, of 48 65 / 79, of 64 94 / 79. 60000 rows of 4: 25 / 34 and
// 19 / 26; 27280: 19 / 18 and 18 / 15.
constexpr int64_t kManyRows = 32768;
constexpr int64_t kNarrowLn = 28, kNarrowRms = 64;
// (that form: 8 threads per row, then one per value or pair, in one grid each)
inline bool narrow(int64_t rows, int64_t cols, int64_t below, int64_t threads) {
  return cols < below && rows > kManyRows && 8 * rows < int64_t(1) << 32 &&
         threads < int64_t(1) << 32;
}

typedef float v4f __attribute__((ext_vector_type(4)));

// A wave's place in its workgroup: 0 .. kWaves - 1 hold rows, kWaves adds.
// Workgroups that share a CU (256 apart) add on different SIMDs.
__device__ __forceinline__ int role() {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int adder = kWaves - (int)(blockIdx.x >> 8 & 3);
  return w == adder ? kWaves : w > adder ? w - 1 : w;
}

// LDS of the chain: a ring of three chunks of the rows, each row 16 bytes
// longer than its columns (the rows' reads then fall on different banks), and
// the rows' sums.
struct alignas(16) Lds {
  float t[3][kRows][kChunk + 4];
  float sum[kRows];
};

// The LDS writes of all waves are done; global loads may stay in flight
// (__syncthreads would wait for them).
__device__ __forceinline__ void sync() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A row of K floats (or a vector over the columns) as a buffer descriptor:
// reads past its end give zeros, writes past it are dropped; null: all of them.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const float* p, int K) {
  return rowsum::row_rsrc(p, p ? 4 * (int64_t)K : 0);
}
// This lane's four columns of chunk i.
__device__ __forceinline__ v4f get(__amdgpu_buffer_rsrc_t r, int i, int l) {
  return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                     r, 16 * l + i * (4 * kChunk), 0, 0));
}
__device__ __forceinline__ void set(__amdgpu_buffer_rsrc_t r, int i, int l, v4f v) {
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), r,
                                         16 * l + i * (4 * kChunk), 0, 0);
}

// The value is held in registers from here on, neither computed again from
// its operands nor held beside them.
__device__ __forceinline__ void keep(v4f& v) {
  float a = v[0], b = v[1], c = v[2], d = v[3];
  asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
  v = v4f{a, b, c, d};
}
__device__ __forceinline__ void keep(float& v) { asm volatile("" : "+v"(v)); }

// A wave's two rows.
template <int NC>
struct Rows {
  v4f v[2][NC];
};

template <int NC>
__device__ __forceinline__ void load(Rows<NC>& x, __amdgpu_buffer_rsrc_t r0,
                                     __amdgpu_buffer_rsrc_t r1, int l) {
#pragma unroll
  for (int i = 0; i < NC; i++) {
    x.v[0][i] = get(r0, i, l);
    x.v[1][i] = get(r1, i, l);
  }
}

// Serial sums over the columns of the terms v (PASS 0), (v - mu)^2 (PASS 1), v^2 (PASS 2) of the
// workgroup's rows. Waves of role w < kWaves call put_terms, the other add_terms, in the
// same order and with the same barriers; chunk i is written two barriers
// before its adds begin, so that the adder reads on across chunk ends. out[u] =
// the sum of this wave's row u (rows 2w, 2w + 1 of the workgroup). Columns
// past K add +0 terms, which leave a sum that started at +0 as it is. PASS 1
// leaves v - mu in x.
template <int NC, int PASS>
__device__ __forceinline__ void put_terms(Rows<NC>& x, int K, const float (&mu)[2], Lds& s,
                                          int w, float (&out)[2]) {
  const int l = threadIdx.x & 63;
  auto put = [&](int i) {
    const bool in = i * kChunk + 4 * l < K;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      v4f o;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if (PASS == 1) x.v[u][i][e] = x.v[u][i][e] - mu[u];
        const float d = x.v[u][i][e];
        o[e] = PASS == 0 ? d : in ? d * d : 0.f;
      }
      if (PASS == 1) keep(x.v[u][i]);
      *reinterpret_cast<v4f*>(&s.t[i % 3][2 * w + u][4 * l]) = o;
    }
  };
  put(0);
  if (NC > 1) put(1);
  sync();
#pragma unroll
  for (int i = 0; i < NC; i++) {
    if (i + 2 < NC) put(i + 2);
    sync();
    __builtin_amdgcn_sched_barrier(0);
  }
  sync();
#pragma unroll
  for (int u = 0; u < 2; u++) out[u] = s.sum[2 * w + u];
}

template <int NC>
__device__ __forceinline__ void add_terms(Lds& s) {
  const int l = threadIdx.x & 63;
  const int mine = l % kRows;
  // 32-column tiles, the next one read while this one is added, with one wait
  // per tile: an add takes ~5 cycles (the chain's latency) and every other
  // instruction of this wave as long, so a row costs ~1.3 x its columns.
  constexpr int kTiles = kChunk / 32;
  v4f a[2][8];
  auto read = [&](int i, int t, v4f (&d)[8]) {
    const v4f* row = reinterpret_cast<const v4f*>(s.t[i % 3][mine]) + 8 * t;
#pragma unroll
    for (int q = 0; q < 8; q++) d[q] = row[q];
  };
  float acc = 0.f;
  sync();
  read(0, 0, a[0]);
#pragma unroll 1
  for (int i = 0; i < NC; i++) {
#pragma unroll
    for (int t = 0; t < kTiles; t++) {
      // (the tile after the last: of a chunk written before, not added)
      read(t + 1 < kTiles ? i : i + 1, (t + 1) % kTiles, a[(t + 1) & 1]);
      __builtin_amdgcn_s_waitcnt(15 | 3 << 14 | 7 << 4 | 8 << 8);  // the tile's own reads
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 8; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc = acc + a[t & 1][q][e];
      __builtin_amdgcn_sched_barrier(0);
    }
    sync();
  }
  if (l < kRows) s.sum[l] = acc;
  sync();
}

// Calls f(integral_constant NC) with the fewest chunks (of 2, 4, 6, .. 12)
// that hold K columns: the adder walks NC chunks whatever K is. us with 4, 8 or
// 12 chunks and so: layernorm at 27280 rows of 1536 86.7, 71.8, of 512 33.5,
// 24.4 (the two-kernel form 142.7, 58.5); norm + quantizer + GEMM of 768 x 1536
// 33.4, 30.2. A form of one chunk ran three times as long as that of two.
template <class F>
auto for_cols(int64_t K, F f) {
  if (K <= 2 * kChunk) return f(std::integral_constant<int, 2>{});
  if (K <= 4 * kChunk) return f(std::integral_constant<int, 4>{});
  if (K <= 6 * kChunk) return f(std::integral_constant<int, 6>{});
  if (K <= 8 * kChunk) return f(std::integral_constant<int, 8>{});
  if (K <= 10 * kChunk) return f(std::integral_constant<int, 10>{});
  return f(std::integral_constant<int, 12>{});
}

}  // namespace rowblock
}  // namespace sdq
