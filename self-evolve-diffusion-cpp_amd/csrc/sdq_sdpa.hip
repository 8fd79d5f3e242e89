// Scaled dot-product attention over packed keys and values (gfx950), the
// form of sdq_sdpa that has scratch memory (src/model/blocks.cpp:112-199,
// non-causal, head_dim 128): every fp32 product as three fp16 MFMA products
// of power-of-two-scaled parts (x = hi + lo; hi.hi + hi.lo + lo.hi, ~2^-22
// relative), an online softmax, fp32 accumulation. Its error against float64
// is below that of the form without scratch (sdq_glue.hip, whose P.V is split
// into bf16 parts): 2.0e-6 against 4.8e-6 of the output's norm at 27280
// tokens, 3.5e-7 against 3.8e-6 at 157 queries x 768 keys.
//
// What bounds it: the matrix cores, and with random operands their power
// (12 Lq Lk 128 operations per head; a library bf16 GEMM reaches 1.37 PFLOP/s
// on this card, a bare loop of these MFMAs with the same LDS reads 1.66). The
// other form splits and transposes every K / V block again for each 256
// queries, a third of its VALU work; here one pass does it once, in the order
// the MFMAs read, so that LDS-DMAs move the blocks as they are and the loop
// holds MFMAs, LDS reads and the softmax only. 27280^2, 24 heads: 30.2 ms
// without, 19.5-20.3 ms with it (0.25 ms of that the packing); MFMAs 16x16x32:
// 32x32x16 ones took 20.7 ms (fewer accumulator bits switch, a higher clock).
#include "sdq_internal.h"
#include "sdq_device.h"
#include "sdq_sdpa_plan.h"

#pragma clang fp contract(off)

namespace sdq {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v2s __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

using sdpa::kHd;
using sdpa::kKB;
using sdpa::kQ;
using sdpa::kRec;
using sdpa::Plan;
constexpr int kRecV = 16384;         // V's offset in it
constexpr int kPart = 8192;          // one part (hi or lo) of K or V
constexpr int kWaves = 8;
static_assert(kQ == 32 * kWaves);
constexpr int kRing = 4;             // blocks of K and of V in LDS
// Operands are scaled by powers of two so that the largest element of a key
// block's K, of its V, and of a query row lies in [2^14, 2^15). hi + lo then
// hold 22 bits of an element down to 2^-18 of that largest one and an absolute
// 2^-40 of it below.
constexpr int kTop = 15;
// A row of K or V whose largest element lies 2^kShift or more below its block's
// is scaled up by 2^(a multiple of kShift), its scores or P down by the same, so
// that no key's logits or P v are lost beside another's: a block with such rows
// is uneven. (Errors of the output's scale without and with it: weights of 2^-20
// on V 2^20 larger 1e-3, 6e-6; V of 2^40 and 2^-90 130%, 4e-6; all the weight on
// keys 2^30 shorter than their neighbours 8e-3, 4e-6. Ordinary blocks keep their
// values; 27280 tokens 1% longer, 157 x 768 34.6 -> 35.7 us.)
constexpr int kShift = 8;
// Blocks whose V lies this far below the head's largest are treated like
// uneven ones (their P may be 0 where their weights are not).
constexpr int kFar = 60;
constexpr int kZeroV = 1 << 20;      // "exponent" of a V block of zeros
constexpr int kMinLogit = -100;      // scales of q.k below 2^this: all logits 0 either way
// V's exponents stop here (a V block all below 2^-95 then holds smaller
// numbers) and the sums l are kept as l 2^-16: l ~ 2^(15 - e_v) stays a normal
// float over all exponents.
constexpr int kMinV = -110;
constexpr int kSumExp = 16;

// The exponent that scales a largest magnitude into [2^14, 2^15) (x = 0: any)
__device__ __forceinline__ int top_exp(float x) {
  return (x > 0.f ? __builtin_amdgcn_frexp_expf(x) : 0) - kTop;
}
// max(m, |x|) over finite x: an infinity or NaN reaches its own products only
__device__ __forceinline__ float amax_finite(float m, float x) {
  const float a = fabsf(x);
  return a <= 3.402823466e38f ? fmaxf(m, a) : m;
}

// max / sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48 of a query, in all
// of them
template <class F>
__device__ __forceinline__ float quad16(float v, F f) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float quad16_max(float v) {
  return quad16(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float quad16_sum(float v) {
  return quad16(v, [](float a, float b) { return a + b; });
}

// One workgroup per (key block, head, sequence): K scaled by the block's
// power of two and split into fp16 parts, V the same, both in
// the order the MFMA operands are read (16 bytes per lane):
//   K [part][32-dim step d][16-key tile kt][lane]: key 16 kt + lane % 16,
//     dims 32 d + 8 (lane / 16) + 0..7
//   V [part][16-dim tile dt][lane]: dim 16 dt + lane % 16, keys
//     16 (m / 4) + 4 (lane / 16) + m % 4, m = 0..7
// Keys past Lk are zeros. exps: K's exponent and 2 e + (uneven) with V's e
// (kZeroV in the place of 2 e: zeros); shifts: V's keys', then K's, in units of
// kShift, a byte each. HBM-bound: 8 bytes read and 8
// written per (key, dim) pair of K and V.
__global__ void __launch_bounds__(256)
sdpa_pack_kernel(const float* __restrict__ K, int64_t ldk, const float* __restrict__ V,
                 int64_t ldv, int64_t Lk, int nkb, char* __restrict__ packed,
                 int2* __restrict__ exps, uint8_t* __restrict__ shifts) {
  __shared__ __attribute__((aligned(16))) char buf[kRec];
  __shared__ __attribute__((aligned(16))) float rows[2][kKB];  // V's, K's largest magnitudes
  const int t = threadIdx.x;
  const int kb = blockIdx.x, head = blockIdx.y;
  const int64_t seq = blockIdx.z;
  const int64_t rec = (seq * gridDim.y + head) * nkb + kb;
  const float* kp = K + seq * Lk * ldk + (int64_t)head * kHd;
  const float* vp = V + seq * Lk * ldv + (int64_t)head * kHd;
  // 4 dims (float4 q4 of a row) of 4 keys each: K's keys 8 i + r, V's 4 r + i
  const int q4 = t & 31, r = t >> 5;
  float4 a[4];
  float v[4][4], mk[4], mv[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int64_t kr = (int64_t)kb * kKB + 8 * i + r, vr = (int64_t)kb * kKB + 4 * r + i;
    a[i] = kr < Lk ? *reinterpret_cast<const float4*>(kp + kr * ldk + 4 * q4)
                   : float4{0.f, 0.f, 0.f, 0.f};
    const float4 x = vr < Lk ? *reinterpret_cast<const float4*>(vp + vr * ldv + 4 * q4)
                             : float4{0.f, 0.f, 0.f, 0.f};
    v[i][0] = x.x, v[i][1] = x.y, v[i][2] = x.z, v[i][3] = x.w;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    mk[i] = amax_finite(amax_finite(0.f, a[i].x), a[i].y);
    mk[i] = amax_finite(amax_finite(mk[i], a[i].z), a[i].w);
    mv[i] = 0.f;
#pragma unroll
    for (int c = 0; c < 4; c++) mv[i] = amax_finite(mv[i], v[i][c]);
  }
  // four rows' maxima over 32 lanes: each lane goes on with two, then with one
  // of them, row mine
  const bool b0 = t & 1, b1 = t & 2;
  const int mine = 2 * (t & 1) + (t >> 1 & 1);
  auto row_max = [&](const float (&m)[4]) {
    float m0 = fmaxf(b0 ? m[2] : m[0], __shfl_xor(b0 ? m[0] : m[2], 1));
    const float m1 = fmaxf(b0 ? m[3] : m[1], __shfl_xor(b0 ? m[1] : m[3], 1));
    m0 = fmaxf(b1 ? m1 : m0, __shfl_xor(b1 ? m0 : m1, 2));
#pragma unroll
    for (int d = 4; d < 32; d *= 2) m0 = fmaxf(m0, __shfl_xor(m0, d));
    return m0;
  };
  const float rv = row_max(mv), rk = row_max(mk);
  if (q4 < 4) rows[0][4 * r + mine] = rv, rows[1][8 * mine + r] = rk;
  __syncthreads();
  float top = 0.f, topk = 0.f;
#pragma unroll
  for (int i = 0; i < kKB; i++) top = fmaxf(top, rows[0][i]), topk = fmaxf(topk, rows[1][i]);
  auto v_exp = [](float m) { return top_exp(m) < kMinV ? kMinV : top_exp(m); };
  const int ek = top_exp(topk), ev = v_exp(top);
  auto v_shift = [&](float m) { return m > 0.f ? (ev - v_exp(m)) & -kShift : 0; };
  auto k_shift = [&](float m) { return m > 0.f ? (ek - top_exp(m)) & -kShift : 0; };
  int sh[4], shk[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
    sh[i] = v_shift(rows[0][4 * r + i]), shk[i] = k_shift(rows[1][8 * i + r]);
  if (t < 64) {
    const float m = rows[t >> 5][t & 31];
    const int sm = t < 32 ? v_shift(m) : k_shift(m);
    shifts[rec * 2 * kKB + t] = (uint8_t)(sm / kShift);
    const int uneven = __ballot(sm > 0) != 0;
    if (t == 0) exps[rec] = int2{ek, (top == 0.f ? kZeroV : 2 * ev) + uneven};
  }
  auto put = [&](char* p, const float y0, const float y1, const float y2, const float y3) {
    const v4h hi = {(_Float16)y0, (_Float16)y1, (_Float16)y2, (_Float16)y3};
    const v4h lo = {(_Float16)(y0 - (float)hi.x), (_Float16)(y1 - (float)hi.y),
                    (_Float16)(y2 - (float)hi.z), (_Float16)(y3 - (float)hi.w)};
    *reinterpret_cast<v4h*>(p) = hi;
    *reinterpret_cast<v4h*>(p + kPart) = lo;
  };
  // The record is put together in LDS and copied out whole. Its 16-byte
  // lane slots are XORed within each 256 bytes (swz) so that the lanes of a
  // wave, which hold different dims of one key, write to different banks.
  auto swz = [](int chunk, int slot) {
    return chunk * 1024 + (slot & 48) * 16 + ((slot & 15) ^ ((slot >> 4) * 4 + (chunk >> 1 & 3))) * 16;
  };
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int key = 8 * i + r;
    put(buf + swz((q4 >> 3) * 2 + (key >> 4), (q4 >> 1 & 3) * 16 + (key & 15)) + (q4 & 1) * 8,
        ldexpf(a[i].x, shk[i] - ek), ldexpf(a[i].y, shk[i] - ek), ldexpf(a[i].z, shk[i] - ek),
        ldexpf(a[i].w, shk[i] - ek));
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int d = 4 * q4 + c;
    put(buf + kRecV + swz(d >> 4, (r & 3) * 16 + (d & 15)) + (r >> 2) * 8,
        ldexpf(v[0][c], sh[0] - ev), ldexpf(v[1][c], sh[1] - ev), ldexpf(v[2][c], sh[2] - ev),
        ldexpf(v[3][c], sh[3] - ev));
  }
  __syncthreads();
  char* dst = packed + rec * kRec;
#pragma unroll
  for (int i = 0; i < kRec / 4096; i++) {
    const int u = i * 256 + t;  // 16-byte slot of the record
    *reinterpret_cast<uint4*>(dst + u * 16) = *reinterpret_cast<const uint4*>(
        buf + (u >> 9) * kPart + swz(u >> 6 & 7, u & 63));
  }
}

struct Parts {
  float* o;    // [seq][slots][256][128]
  float2* ml;  // [seq][slots][256]: (reference, sum), base 2
};

// One MFMA operand of a lane as its high and low parts.
struct Frag {
  uint4 hi, lo;
};
__device__ __forceinline__ v4f mfma_h(const uint4& a, const v8h& b, const v4f& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), b, c, 0, 0, 0);
}
// o / l from a sum kept as l 2^-kSumExp, its exponent applied last (1 / l
// itself may be subnormal)
struct Inv {
  float r;
  int e;
  __device__ __forceinline__ explicit Inv(float l)
      : r(1.f / __builtin_amdgcn_frexp_mantf(l)), e(-__builtin_amdgcn_frexp_expf(l) - kSumExp) {}
  __device__ __forceinline__ float operator()(float o) const { return ldexpf(o * r, e); }
};

// l 2^d: for d below -100 in two steps, since the exponential's 2^d becomes 0
// below the normal numbers, which l 2^d need not be
__device__ __forceinline__ float scale_l(float l, float d) {
  const float half = __builtin_amdgcn_exp2f(0.5f * d);
  return d < -100.f ? l * half * half : l * __builtin_amdgcn_exp2f(d);
}

// Keeps a value's computation where it is written (the compiler would sink it
// past the barrier to its use).
template <class T>
__device__ __forceinline__ void pin(T& v) {
  asm volatile("" : "+v"(v));
}

// a, b as fp16 hi + lo, each part's pair in a dword. neg1 = -1 unknown to the
// compiler: x - hi then stays a multiply-add that reads hi as fp16 and writes
// fp16 (one instruction per low part).
__device__ __forceinline__ void split_pair(float a, float b, float neg1, uint32_t& hi,
                                           uint32_t& lo) {
  hi = __builtin_bit_cast(uint32_t, v2h{(_Float16)a, (_Float16)b});
  pin(hi);  // the low parts read its halves
  const v2h h = __builtin_bit_cast(v2h, hi);
  lo = __builtin_bit_cast(uint32_t, v2h{(_Float16)__builtin_fmaf((float)h.x, neg1, a),
                                        (_Float16)__builtin_fmaf((float)h.y, neg1, b)});
}

__global__ void __launch_bounds__(kWaves * 64)
sdpa_packed_kernel(const float* __restrict__ Q, int64_t ldq, const char* __restrict__ packed,
                   const int2* __restrict__ exps, const uint32_t* __restrict__ shifts,
                   float* __restrict__ O, int64_t ldo, int64_t Lq, int64_t Lk, Plan plan,
                   float scale_log2e, Parts parts) {
  constexpr int QT = 2;            // 16-query tiles per wave
  constexpr int LD = 16 / kWaves;  // a wave's DMAs of one K or V block
  __shared__ __attribute__((aligned(16))) char lds[kRing * kRec];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, h = lane >> 4;
  const int64_t seq = blockIdx.y;
  const float* Qs = Q + seq * Lq * ldq;
  float* Os = O + seq * Lq * ldo;
  const int nkb = plan.nkb;

  // This workgroup's item and key range: consecutive items on one XCD
  // (workgroup b runs on XCD b % 8), so its CUs walk the same head's blocks
  // and share them in the XCD's L2.
  int item, kb0 = 0, kb1 = nkb, slot = -1;
  {
    const bool whole = (int)blockIdx.x < plan.nfull;
    const int c = whole ? blockIdx.x : blockIdx.x - plan.nfull;
    const int total = whole ? plan.nfull : (plan.items - plan.nfull) * plan.splits;
    const int x = c & 7, q8 = total >> 3, r8 = total & 7;
    item = x * q8 + (x < r8 ? x : r8) + (c >> 3);
    if (!whole) {
      if (plan.splits > 1) slot = item;
      kb0 = item % plan.splits * plan.kbs;
      kb1 = kb0 + plan.kbs < nkb ? kb0 + plan.kbs : nkb;
      item = plan.nfull + item / plan.splits;
    }
  }

  const uint32_t lane16 = (uint32_t)lane * 16u;
  const char* ldsp = lds + lane16;
  const uint32_t ldsw =
      __builtin_amdgcn_readfirstlane(dev::lds_addr32(lds)) + (uint32_t)(w * LD) * 1024u;
  const uint32_t voff = lane16 + (uint32_t)(w * LD) * 1024u;
  const int head = item / plan.qgroups, qg = item - head * plan.qgroups;
  const int64_t q0 = (int64_t)qg * kQ + w * (16 * QT);
  const int64_t col = (int64_t)head * kHd;
  const int64_t rec0 = (seq * (plan.items / plan.qgroups) + head) * nkb;
  const int2* ex = exps + rec0;

  // This wave's DMAs: LD of the 16 1 KB-chunks of K(i) or V(i) (block kb0 + i)
  // into ring slot i % kRing; blocks past the range repeat the last one
  // (never used).
  const dev::v4u rs = dev::raw_rsrc(packed + rec0 * kRec, (uint32_t)nkb * (uint32_t)kRec);
  auto soff = [&](int i) { return (uint32_t)(kb0 + i < kb1 ? kb0 + i : kb1 - 1) * kRec; };
  auto slot_k = [&](int i) { return ldsw + (uint32_t)(i & (kRing - 1)) * kRecV; };
  auto slot_v = [&](int i) { return ldsw + (uint32_t)(kRing + (i & (kRing - 1))) * kRecV; };
  auto issue_k = [&](int i) {
#pragma unroll
    for (int c = 0; c < LD; c++)
      dev::dma16<0>(rs, voff, soff(i) + c * 1024u, slot_k(i) + c * 1024u);
  };
  auto issue_v = [&](int i) {
#pragma unroll
    for (int c = 0; c < LD; c++)
      dev::dma16<0>(rs, voff, soff(i) + kRecV + c * 1024u, slot_v(i) + c * 1024u);
  };
  const int n = kb1 - kb0;
  // A wave past the queries moves its share of the blocks and no more (the
  // same waits and barriers as below).
  if (q0 >= Lq) {
    issue_k(0), issue_v(0), issue_k(1), issue_v(1), issue_k(2), issue_v(2), issue_k(3);
    __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(6 * LD));
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(4 * LD));
    asm volatile("s_barrier" ::: "memory");
    issue_k(4);
    for (int i = 0; i < n; i++) {
      __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(3 * LD));
      asm volatile("s_barrier" ::: "memory");
      issue_v(i + 3), issue_k(i + 5);
    }
    __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(0));
    return;
  }
  float neg1 = -1.f;  // for split_pair
  asm volatile("" : "+s"(neg1));
  // Everything the first scores need is asked for at once: block exponents
  // (64 blocks from kb0, one per lane, and the first 64 of all), query rows,
  // and the first DMAs; the other DMAs follow the queries' conversion, whose
  // wait would cover them too.
  int2 ev = ex[kb0 + lane < nkb ? kb0 + lane : nkb - 1];
  const int ev0 = ex[lane < nkb ? lane : nkb - 1].y;
  // The query rows, lane (j, h): dims 32 d + 8 h + 0..7 of query 16 t + j,
  // scaled by 2^-eq and split into fp16 parts
  v8h qh[QT][4], ql[QT][4];
  int eq[QT];
  float4 qrow[QT][8];
#pragma unroll
  for (int t = 0; t < QT; t++) {
    const int64_t qi = q0 + 16 * t + j;
    const float* src = Qs + (qi < Lq ? qi : 0) * ldq + col + 8 * h;  // past Lq: not stored
#pragma unroll
    for (int c = 0; c < 8; c++)
      qrow[t][c] = *reinterpret_cast<const float4*>(src + 32 * (c >> 1) + 4 * (c & 1));
  }
  issue_k(0), issue_v(0), issue_k(1);
#pragma unroll
  for (int t = 0; t < QT; t++) {
    const float4(&qr)[8] = qrow[t];
    float mq = 0.f;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      mq = fmaxf(fmaxf(mq, fabsf(qr[c].x)), fabsf(qr[c].y));
      mq = fmaxf(fmaxf(mq, fabsf(qr[c].z)), fabsf(qr[c].w));
    }
    eq[t] = top_exp(quad16_max(mq));
#pragma unroll
    for (int d = 0; d < 4; d++) {
      uint32_t* hw = reinterpret_cast<uint32_t*>(&qh[t][d]);
      uint32_t* lw = reinterpret_cast<uint32_t*>(&ql[t][d]);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float4& v = qr[2 * d + (e >> 1)];
        split_pair(ldexpf(e & 1 ? v.z : v.x, -eq[t]), ldexpf(e & 1 ? v.w : v.y, -eq[t]), neg1,
                   hw[e], lw[e]);
      }
    }
  }
  issue_v(1), issue_k(2), issue_v(2), issue_k(3);
  // the largest and smallest V exponents of the head's blocks (16 bits each,
  // the smallest negated); a block of zeros takes the smallest
  auto range = [](int y) {
    return y >= kZeroV ? v2s{-1000, -1000} : v2s{(short)(y >> 1), (short)-(y >> 1)};
  };
  v2s vr = range(ev0);
  for (int k = lane + 64; k < nkb; k += 64) vr = __builtin_elementwise_max(vr, range(ex[k].y));
#pragma unroll
  for (int d = 1; d < 64; d *= 2)
    vr = __builtin_elementwise_max(
        vr, __builtin_bit_cast(v2s, __shfl_xor(__builtin_bit_cast(int, vr), d)));
  const int vmin = vr.x == -1000 ? 0 : -vr.y, vfar = vr.x - kFar;
  // the partial block, if this range ends with it (else never reached)
  const int rem = (int)(Lk % kKB);
  const int last = rem && kb1 == nkb ? n - 1 : -1;
  // 64 blocks' exponents, which of them are uneven or far below, and at which
  // the loop's common path ends: those, the partial block, and the next 64's
  // first
  uint64_t odd, stops;
  auto decode_ev = [&](int i) {
    const bool zero = ev.y >= kZeroV, uneven = ev.y & 1;
    ev.y = zero ? vmin : ev.y >> 1;
    odd = __ballot(uneven || ev.y < vfar);
    stops = odd | 1 | (last >= i && last < i + 64 ? (uint64_t)1 << (last & 63) : 0);
  };
  auto load_ev = [&](int i) {
    const int k = kb0 + i + lane;
    ev = ex[k < nkb ? k : nkb - 1];
    decode_ev(i);
  };
  decode_ev(0);
  auto is_odd = [&](int i) { return (odd >> (i & 63) & 1) != 0; };
  // the V (v = 0) or K shifts of keys 16 kt + 4 h .. + 3 of block i, a byte each
  auto key_shifts = [&](int i, int v, int kt) {
    return shifts[(rec0 + kb0 + i) * (2 * kKB / 4) + 8 * v + 4 * kt + h];
  };
  auto shift_of = [](uint32_t u, int r) { return (int)(u >> 8 * r & 255) * kShift; };
  auto kfrag = [&](int i, int c) {
    const char* p = ldsp + (i & (kRing - 1)) * kRecV + c * 1024;
    return Frag{*reinterpret_cast<const uint4*>(p), *reinterpret_cast<const uint4*>(p + kPart)};
  };
  auto vfrag = [&](int i, int c) {
    const char* p = ldsp + (kRing + (i & (kRing - 1))) * kRecV + c * 1024;
    return Frag{*reinterpret_cast<const uint4*>(p), *reinterpret_cast<const uint4*>(p + kPart)};
  };
  // scores of a block: S^T tile [kt][t], keys 16 kt + 4 h + r of query 16 t + j
  struct Scores {
    v4f s[2][QT];
  };
  v4f acc[8][QT];  // O^T tile [dt][t]: dims 16 dt + 4 h + r of query 16 t + j
#pragma unroll
  for (int d = 0; d < 8; d++)
#pragma unroll
    for (int t = 0; t < QT; t++) acc[d][t] = v4f{};
  // R: the reference exponent of a query; P = 2^(s + e_v - R) with the base-2
  // logit s and V's exponent e_v (its block's, less the key's shift), so that
  // P V~ (V~ = V 2^-e_v) sums to 2^-R sum 2^s V. R follows max(s + e_v), kept in
  // [R + 7, R + 15]: P is then at most 2^15, its fp16 parts keep 22 bits down
  // to 2^-10 of the largest so far (and an absolute 2^-32 of it below), and the
  // accumulators are rarely rescaled. l = 2^(-R - kSumExp) sum 2^s: the sum of a
  // block's P with its e_v taken out, but from the logits again where keys of
  // a block differ in e_v or P may have become 0 beside V larger elsewhere.
  float R[QT], lsum[QT], sq[QT], off[QT];
#pragma unroll
  for (int t = 0; t < QT; t++) R[t] = -INFINITY, lsum[t] = 0.f;
  auto mask = [&](Scores& sc) {
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (16 * kt + 4 * h + r >= rem)
#pragma unroll
          for (int t = 0; t < QT; t++) sc.s[kt][t][r] = -INFINITY;
  };
  auto max4 = [&](float x, const v4f& v) {
    x = fmaxf(fmaxf(x, v[0]), v[1]);
    return fmaxf(fmaxf(x, v[2]), v[3]);
  };
  auto raise = [&](const float* mb, float e) {
#pragma unroll
    for (int t = 0; t < QT; t++) {
      const bool u = mb[t] > R[t] + 15.f;
      const float rn = u ? mb[t] - 7.f : R[t];
      const float alpha = u ? __builtin_amdgcn_exp2f(R[t] - rn) : 1.f;
      lsum[t] = u ? scale_l(lsum[t], R[t] - rn) : lsum[t];
      R[t] = rn;
      off[t] = e - rn;
#pragma unroll
      for (int d = 0; d < 8; d++) acc[d][t] *= alpha;
    }
  };

  // the scale of q.k in base 2
  auto logit_scale = [&](int t, int kx) {
    return ldexpf(scale_log2e, max(eq[t] + kx, kMinLogit));
  };
  // An odd block's scores, down by its keys' shifts
  auto shift_keys = [&](Scores& sc, int i) {
    const int kx = __builtin_amdgcn_readlane(ev.x, i & 63);
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      const uint32_t u = key_shifts(i, 0, kt), uk = key_shifts(i, 1, kt);
#pragma unroll
      for (int t = 0; t < QT; t++) {
        const float up = -1.f / logit_scale(t, kx);
#pragma unroll
        for (int r = 0; r < 4; r++)
          sc.s[kt][t][r] =
              fmaf((float)shift_of(u, r), up, ldexpf(sc.s[kt][t][r], -shift_of(uk, r)));
      }
    }
  };
  // An odd block's part of l, from its shifted scores (whose sq and off are set)
  auto add_l = [&](const Scores& sc, int i) {
    const int e_v = __builtin_amdgcn_readlane(ev.y, i & 63);
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      const uint32_t u = key_shifts(i, 0, kt);
#pragma unroll
      for (int t = 0; t < QT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          lsum[t] += __builtin_amdgcn_exp2f(fmaf(sc.s[kt][t][r], sq[t], off[t]) +
                                            (float)(shift_of(u, r) - e_v - kSumExp));
    }
  };

  Frag fr[4];
  // K(0) has landed (newer DMAs may be in flight), then V(0) and K(1)
  __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(6 * LD));
  asm volatile("s_barrier" ::: "memory");
  Scores st, st2;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int d = c >> 1, kt = c & 1;
    const Frag f = kfrag(0, c);
#pragma unroll
    for (int t = 0; t < QT; t++) st.s[kt][t] = mfma_h(f.hi, qh[t][d], d ? st.s[kt][t] : v4f{});
#pragma unroll
    for (int t = 0; t < QT; t++) st.s[kt][t] = mfma_h(f.hi, ql[t][d], st.s[kt][t]);
#pragma unroll
    for (int t = 0; t < QT; t++) st.s[kt][t] = mfma_h(f.lo, qh[t][d], st.s[kt][t]);
  }
  if (last == 0) mask(st);
  if (is_odd(0)) shift_keys(st, 0);
  {
    float mb[QT];
#pragma unroll
    for (int t = 0; t < QT; t++) {
      sq[t] = logit_scale(t, __builtin_amdgcn_readlane(ev.x, 0));
      mb[t] = fmaf(quad16_max(max4(max4(-INFINITY, st.s[0][t]), st.s[1][t])), sq[t],
                   (float)__builtin_amdgcn_readlane(ev.y, 0));
    }
    raise(mb, (float)__builtin_amdgcn_readlane(ev.y, 0));
    if (is_odd(0)) add_l(st, 0);
  }
  __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(4 * LD) & ~(15 << 8));
  asm volatile("s_barrier" ::: "memory");
  issue_k(4);
  fr[0] = kfrag(1, 0);
  fr[1] = kfrag(1, 1);

  // Block i, whose scores sc, scale sq and offset off = e_v - R are known: the next
  // block's scores on the matrix cores beside this block's exponentials,
  // then P.V beside the next block's maximum. Every group of MFMAs is fenced
  // with its share of the other work, and operands are read two steps
  // ahead, so the MFMA pipe does not wait for either.
  auto step = [&](int i, const Scores& sc, Scores& nx) {
    v8h ph[QT], pl[QT];
    uint32_t* phw = reinterpret_cast<uint32_t*>(ph);
    uint32_t* plw = reinterpret_cast<uint32_t*>(pl);
    float x0[QT / 2], x1[QT / 2], ps[QT];
#pragma unroll
    for (int t = 0; t < QT; t++) ps[t] = 0.f;
    const int e_v = __builtin_amdgcn_readlane(ev.y, i & 63);
    const int i1 = i + 1;
    const bool special = stops >> (i1 & 63) & 1;
    const int e_l = is_odd(i) ? -1000 : -kSumExp - e_v;  // odd: add_l has been there
    // pair u of step c: elements 2 e, 2 e + 1 (of 8) of query tile t
    auto elem = [&](int c, int u, int k, int& t, int& e) {
      const int pi = c * (QT / 2) + u;
      t = pi >> 2, e = pi & 3;
      return __builtin_amdgcn_exp2f(fmaf(sc.s[e >> 1][t][2 * (e & 1) + k], sq[t], off[t]));
    };
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const int d = c >> 1, kt = c & 1;
      const Frag f = fr[c & 3];
      fr[(c + 2) & 3] = c + 2 < 8 ? kfrag(i + 1, c + 2) : vfrag(i, c + 2 - 8);
      int t0, e0;
#pragma unroll
      for (int t = 0; t < QT; t++)
        nx.s[kt][t] = mfma_h(f.hi, qh[t][d], d ? nx.s[kt][t] : v4f{});
#pragma unroll
      for (int u = 0; u < QT / 2; u++) {
        x0[u] = elem(c, u, 0, t0, e0);
        pin(x0[u]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < QT; t++) nx.s[kt][t] = mfma_h(f.hi, ql[t][d], nx.s[kt][t]);
#pragma unroll
      for (int u = 0; u < QT / 2; u++) {
        x1[u] = elem(c, u, 1, t0, e0);
        ps[t0] += x0[u];
        pin(x1[u]), pin(ps[t0]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < QT; t++) nx.s[kt][t] = mfma_h(f.lo, qh[t][d], nx.s[kt][t]);
#pragma unroll
      for (int u = 0; u < QT / 2; u++) {
        const int pi = c * (QT / 2) + u;
        ps[pi >> 2] += x1[u];
        // P = fp16 hi + fp16 lo, two keys per dword
        split_pair(x0[u], x1[u], neg1, phw[pi], plw[pi]);
        pin(plw[pi]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // own DMAs of V(i+1) and K(i+2) have landed; after the barrier
    // everyone's have, and K(i+1), V(i-1) have been read by all
    __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(3 * LD));
    asm volatile("s_barrier" ::: "memory");
    if (special) {
      if ((i1 & 63) == 0) load_ev(i1);
      if (i1 == last) mask(nx);
      if (i1 < n && is_odd(i1)) shift_keys(nx, i1);
    }
    const uint32_t sv = soff(i + 3) + kRecV, sk = soff(i + 5);
    const uint32_t dv = slot_v(i + 3), dk = slot_k(i + 5);
    float ml[QT], vx = 0.f;
    int kx = 0;
    bool up = false;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const Frag f = fr[c & 3];
      fr[(c + 2) & 3] = c + 2 < 8 ? vfrag(i, c + 2) : kfrag(i + 2, c + 2 - 8);
      // O^T += V^T . P^T: V_hi.P_hi + V_hi.P_lo + V_lo.P_hi
#pragma unroll
      for (int t = 0; t < QT; t++) acc[c][t] = mfma_h(f.hi, ph[t], acc[c][t]);
      // LD DMAs of V, then LD of K: LD / 2 of either per step
      if (c < 4) {
#pragma unroll
        for (int u = 0; u < LD / 2; u++) {
          const uint32_t o = (uint32_t)((c & 1) * (LD / 2) + u) * 1024u;
          dev::dma16<0>(rs, voff, (c < 2 ? sv : sk) + o, (c < 2 ? dv : dk) + o);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < QT; t++) acc[c][t] = mfma_h(f.hi, pl[t], acc[c][t]);
      if (c >= 2 && c < 4) {
#pragma unroll
        for (int t = 0; t < QT; t++) {
          ml[t] = max4(c == 2 ? -INFINITY : ml[t], nx.s[c - 2][t]);
          pin(ml[t]);
        }
      }
      if (c == 1) {
#pragma unroll
        for (int t = 0; t < QT; t++) {
          lsum[t] += ldexpf(ps[t], e_l);
          pin(lsum[t]);
        }
      }
      if (c == 4) {
        kx = __builtin_amdgcn_readlane(ev.x, i1 & 63);
        vx = (float)__builtin_amdgcn_readlane(ev.y, i1 & 63);
#pragma unroll
        for (int t = 0; t < QT; t++) {
          sq[t] = logit_scale(t, kx);
          pin(sq[t]);
        }
      }
      if (c == 6) {
#pragma unroll
        for (int t = 0; t < QT; t++) {
          up = up || ml[t] > R[t] + 15.f;
          off[t] = vx - R[t];
          pin(off[t]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < QT; t++) acc[c][t] = mfma_h(f.lo, ph[t], acc[c][t]);
      if (c == 5) {
#pragma unroll
        for (int t = 0; t < QT; t++) {
          ml[t] = fmaf(quad16_max(ml[t]), sq[t], vx);
          pin(ml[t]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (i1 < n && (__ballot(up) | (odd >> (i1 & 63) & 1))) {  // (past the end: a repeated block)
      raise(ml, vx);
      if (is_odd(i1)) add_l(nx, i1);
    }
  };
  for (int i = 0;;) {
    step(i, st, st2);
    if (++i == n) break;
    step(i, st2, st);
    if (++i == n) break;
  }

  const int64_t nslots = (int64_t)(plan.items - plan.nfull) * plan.splits;
#pragma unroll
  for (int t = 0; t < QT; t++) {
    const float ltot = quad16_sum(lsum[t]);
    const int64_t qi = q0 + 16 * t + j;
    if (slot >= 0) {
      const int64_t row = (seq * nslots + slot) * kQ + w * (16 * QT) + 16 * t + j;
      float* dst = parts.o + row * kHd + 4 * h;
#pragma unroll
      for (int d = 0; d < 8; d++) *reinterpret_cast<v4f*>(dst + 16 * d) = acc[d][t];
      if (h == 0) parts.ml[row] = float2{R[t], ltot};
    } else if (qi < Lq) {
      const Inv inv(ltot);
      float* dst = Os + qi * ldo + col + 4 * h;
#pragma unroll
      for (int d = 0; d < 8; d++)
        *reinterpret_cast<v4f*>(dst + 16 * d) =
            v4f{inv(acc[d][t][0]), inv(acc[d][t][1]), inv(acc[d][t][2]), inv(acc[d][t][3])};
    }
  }
  // the repeated blocks' DMAs must land before the LDS is given back
  __builtin_amdgcn_s_waitcnt(dev::waitcnt_vm(0));
}

// An item's shares combined: out = sum_s w_s o_s / sum_s w_s l_s, w_s =
// 2^(R_s - max R). One thread per 4 dims of a query.
__global__ void __launch_bounds__(256)
sdpa_combine_kernel(Plan plan, Parts parts, int64_t Lq, float* __restrict__ O, int64_t ldo) {
  const int it = blockIdx.x;  // item nfull + it
  const int64_t seq = blockIdx.z;
  const int q = blockIdx.y * 8 + (threadIdx.x >> 5), d = 4 * (threadIdx.x & 31);
  const int item = plan.nfull + it;
  const int head = item / plan.qgroups, qg = item - head * plan.qgroups;
  const int64_t qi = (int64_t)qg * kQ + q;
  if (qi >= Lq) return;
  const int S = plan.splits;
  const int64_t row = (seq * (plan.items - plan.nfull) + it) * S * kQ + q;
  const float2* ml = parts.ml + row;
  const float* op = parts.o + row * kHd + d;
  float mx = -INFINITY, mn = INFINITY;
  for (int s = 0; s < S; s++) mx = fmaxf(mx, ml[s * kQ].x), mn = fminf(mn, ml[s * kQ].x);
  float lt = 0.f;
  float4 o = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < S; s++) {
    const float2 m = ml[s * kQ];
    const float wt = __builtin_amdgcn_exp2f(m.x - mx);
    lt += wt * m.y;
    const float4 v = *reinterpret_cast<const float4*>(op + (int64_t)s * kQ * kHd);
    o.x += wt * v.x;
    o.y += wt * v.y;
    o.z += wt * v.z;
    o.w += wt * v.w;
  }
  if (mx - mn > 100.f) {
    lt = 0.f;
    for (int s = 0; s < S; s++) lt += scale_l(ml[s * kQ].y, ml[s * kQ].x - mx);
  }
  const Inv inv(lt);
  *reinterpret_cast<float4*>(O + (seq * Lq + qi) * ldo + (int64_t)head * kHd + d) =
      float4{inv(o.x), inv(o.y), inv(o.z), inv(o.w)};
}

}  // namespace

int64_t sdpa_packed_bytes(int64_t Lq, int64_t Lk, int heads, int batch, int cu_count) {
  return sdpa::scratch_bytes(Lq, Lk, heads, batch, cu_count);
}

hipError_t launch_sdpa_packed(const float* q, int64_t ldq, const float* k, int64_t ldk,
                              const float* v, int64_t ldv, float* out, int64_t ldo, int64_t Lq,
                              int64_t Lk, int heads, hipStream_t s, int batch, void* scratch,
                              int64_t scratch_bytes, int cu_count) {
  if (Lq <= 0 || batch <= 0) return hipSuccess;
  if (Lk <= 0 || heads <= 0 || heads > 65535 || batch > 65535 || !scratch)
    return hipErrorInvalidValue;
  const float scale_log2e = (1.f / sqrtf((float)kHd)) * 1.4426950408889634f;
  const sdpa::Chunk ch = sdpa::chunk(Lq, Lk, heads, batch, cu_count);
  char* packed = static_cast<char*>(scratch);
  for (int b0 = 0; b0 < batch; b0 += ch.seqs)
    for (int h0 = 0; h0 < heads; h0 += ch.heads) {
      const int nb = batch - b0 < ch.seqs ? batch - b0 : ch.seqs;
      const int nh = heads - h0 < ch.heads ? heads - h0 : ch.heads;
      const Plan p = sdpa::launch_plan(Lq, Lk, nh, cu_count);
      const sdpa::Layout l = sdpa::layout(p, nh, nb);
      if (l.bytes > scratch_bytes) return hipErrorInvalidValue;
      int2* exps = reinterpret_cast<int2*>(packed + l.exps);
      uint8_t* shifts = reinterpret_cast<uint8_t*>(packed + l.shifts);
      const Parts parts{reinterpret_cast<float*>(packed + l.o),
                        reinterpret_cast<float2*>(packed + l.ml)};
      const int64_t col = (int64_t)h0 * kHd;
      const float* qb = q + b0 * Lq * ldq + col;
      float* ob = out + b0 * Lq * ldo + col;
      hipLaunchKernelGGL(sdpa_pack_kernel, dim3((unsigned)p.nkb, (unsigned)nh, (unsigned)nb),
                         dim3(256), 0, s, k + b0 * Lk * ldk + col, ldk, v + b0 * Lk * ldv + col,
                         ldv, Lk, p.nkb, packed, exps, shifts);
      const int64_t shares = (int64_t)(p.items - p.nfull) * p.splits;
      hipLaunchKernelGGL(sdpa_packed_kernel, dim3((unsigned)(p.nfull + shares), (unsigned)nb),
                         dim3(kWaves * 64), 0, s, qb, ldq, packed, exps,
                         reinterpret_cast<const uint32_t*>(shifts), ob, ldo, Lq, Lk,
                         p, scale_log2e, parts);
      if (p.splits > 1)
        hipLaunchKernelGGL(sdpa_combine_kernel,
                           dim3((unsigned)(p.items - p.nfull), kQ / 8, (unsigned)nb), dim3(256),
                           0, s, p, parts, Lq, ob, ldo);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}

}  // namespace sdq
