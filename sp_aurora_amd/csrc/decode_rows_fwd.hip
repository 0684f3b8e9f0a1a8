// Attention of up to 16 query rows over a K/V whose rows lie back to back (the decode step of a server that keeps a cache per head, drafted tokens that
// are checked): the block forward of sp_aurora/intel_flash_attn.py:233-296, where the work is reading K and V once.
//
// Both contractions run on v_mfma_f32_16x16x32, whose 16 columns are the query rows, and nothing goes through LDS before the end:
//   S^T = K Q^T    a lane holds 8 dims of one key, as 16 bytes of its row come from memory (of e4m3 keys 16 dims, for two steps);
//   O^T += V^T P^T a lane holds 8 keys of one dim.  It loads the pieces of D / 16 dims of 8 keys, whole rows side by side across 16 lanes, and
//                  transposes them in its own registers (v_perm: one per two elements).  Which 8 keys a group of 16 lanes takes is free as
//                  long as P has the same: those whose scores the first product left in it.
// A lane owns one query row (lane % 16) in S^T, P^T and O^T alike: the running maximum and sum are per-lane values.  The waves of a
// workgroup take every kWaves-th tile of 32 keys, each with a state of its own, and add up through LDS at the end.
// Up to three rows keep their weights in fp32, as three terms of the element type, of bf16 beside e4m3 values (weight_terms).
//
// Grid: x = batch * head, y = key chunk (the key split of the caller: chunk y writes rows y * Sq .. of the result tensors it is given).
// Bound: HBM.  A key's row is requested in pieces of 64 bytes and 16 keys at a time, which is as good as whole rows only where rows lie back to
// back (spa_rows16_takes).
#include <type_traits>

#include "spa_common.h"
#include "spa_host.h"

namespace {

template <typename T>
struct Mma16x16;
template <>
struct Mma16x16<__bf16> {
  static __device__ __forceinline__ f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ unsigned widen(unsigned x, bool hi) {  // two e4m3 bytes (exact)
    return hi ? __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.0f, true))
              : __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.0f, false));
  }
};
template <>
struct Mma16x16<_Float16> {
  static __device__ __forceinline__ f32x4 run(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ unsigned widen(unsigned x, bool hi) {
    return hi ? __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(x, 1.0f, true))
              : __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(x, 1.0f, false));
  }
};

// 4, 8 or 16 bytes of a buffer (offsets past its end give zeros).
template <int DW>
struct Words {
  unsigned w[DW];
};
template <int DW, int AUX>
__device__ __forceinline__ Words<DW> load_words(__amdgpu_buffer_rsrc_t rs, unsigned off) {
  Words<DW> r;
  if constexpr (DW == 4) {
    const u32x4 x = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, AUX));
#pragma unroll
    for (int i = 0; i < 4; ++i) r.w[i] = x[i];
  } else if constexpr (DW == 2) {
    const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, AUX));
#pragma unroll
    for (int i = 0; i < 2; ++i) r.w[i] = x[i];
  } else {
    r.w[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, AUX);
  }
  return r;
}

// The weights of up to three rows are the sum of three terms of the element type, none above that of the largest score (so that large values do not overflow
// under it).  bf16 terms have fp32's range and hold all 24 bits.  fp16's end at 2^-24, so there the largest weight is 2^15 and the terms beside the first, which
// hold 2^-10 of it at most, are 2^11 times as large as what they stand for: 24 bits down to 2^-27 of the largest weight, steps of 2^-50 of it below.  A weight whose
// first term would round to 0 has the smallest one there and the difference in the others, so that an infinity in V under it is one in the result.
// More rows round their weights once, as the kernels for long rows do, and the reference may be 2^8 too low.
constexpr int kRowsInFp32 = 3;
constexpr int weight_terms(int rows) { return rows <= kRowsInFp32 ? 3 : 1; }
template <typename T, int TERMS>
struct WeightRange {
  static constexpr bool half = std::is_same<T, _Float16>::value;
  static constexpr float slack = TERMS > 1 ? 0.f : 8.f;            // log2 of what a score may exceed the reference by
  static constexpr float up = !half ? 0.f : TERMS > 1 ? 15.f : 7.f;        // log2 of the weight of a score at the reference
  static constexpr bool scaled = half && TERMS > 1;
  static constexpr float later = scaled ? 0x1p11f : 1.f;                   // of the terms beside the first
  // what the first term is rounded from: x, or the smallest fp16 number where 0 < x < that
  static __device__ __forceinline__ float first(float x) { return scaled ? __builtin_amdgcn_fmed3f(x, x * 0x1p102f, 0x1p-24f) : x; }
};

template <int D, int kWaves>
struct DecodeCfg {
  static constexpr int PITCH = D + 4;                        // floats of a row in LDS
  static constexpr int REC = 16 * PITCH + 32;                // what a wave leaves: rows, then maxima and sums
  static constexpr int SMEM = kWaves * REC * 4;
};

// NT: the loads carry the non-temporal hint.
template <typename T, int D, bool KV8, int TERMS, int kWaves, bool NT>
__global__ void __launch_bounds__(kWaves * 64) rows16_fwd_kernel(const FwdParams p) {
  constexpr int AUX = NT ? 2 : 0;
  // (e4m3 values are as exact in bf16: weights of several terms have fp32's range there, whatever the type of the queries)
  typedef typename std::conditional<KV8 && (TERMS > 1), __bf16, T>::type PT;
  typedef Mma16<PT> MP;
  typedef Mma16x16<PT> MMP;
  typedef typename MP::frag pfrag;
  typedef Mma16<T> M;
  typedef Mma16x16<T> MM;
  typedef typename M::frag frag;
  typedef DecodeCfg<D, kWaves> C;
  typedef WeightRange<PT, TERMS> W;
  constexpr int KESZ = KV8 ? 1 : 2;
  constexpr int NK = D * KESZ / 64;        // 16-byte loads of a key's row by the four lanes that share it
  constexpr int DL = D / 16;               // dims of V per lane
  constexpr int VW = DL * KESZ / 4;        // their 4-byte words
  // Terms beside the first have sums of their own, for their scale and for V's infinities (e4m3 has neither): where V holds one these sums are no numbers, and
  // the first term's sum is the result.
  constexpr bool REST = TERMS > 1 && !KV8;
  extern __shared__ __align__(16) unsigned char smem[];
  float* const sm = (float*)smem;

  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
  // Workgroups go to the 8 XCDs round robin.  Where a key row is half a cache line (64 e4m3 elements), the rows of two heads side by side share every
  // line: those heads are given to workgroups 8 apart, which run on one XCD at about the same time.
  int bh = blockIdx.x;
  if (D * KESZ < 128 && (gridDim.x & 7) == 0) bh = (bh & 7) * (int)(gridDim.x >> 3) + (bh >> 3);
  const int b = bh / p.H, h = bh - b * p.H, z = blockIdx.y;
  const int k0 = z * p.Sk, k1 = k0 + (z == p.P - 1 ? p.sk_last : p.Sk), nq = p.Sq;

  // the row's queries as operands: element e of step s is the dim that element e of the lane's K operand of that step holds
  frag qf[D / 32];
  {
    const T* const qp = (const T*)p.q + b * p.qs.b + h * p.qs.h + (int64_t)(n < nq ? n : nq - 1) * p.qs.s;
    const unsigned flip = p.negq ? 0x80008000u : 0u;
#pragma unroll
    for (int s = 0; s < D / 32; ++s) {
      u32x4 y = *(const u32x4*)(qp + (KV8 ? 64 * (s / 2) + 16 * g + 8 * (s % 2) : 32 * s + 8 * g));
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] ^= flip;
      qf[s] = as_frag<frag>(y);
    }
  }
  const float c = p.scale_log2 * (KV8 ? p.k_scale[bh] : 1.f);

  // descriptors that end with this chunk's last row: rows past it read as zero and are masked below
  const unsigned krow_b = (unsigned)(p.ks.s * KESZ), vrow_b = (unsigned)(p.vs.s * KESZ);
  const char* const kp = (const char*)p.k + (b * p.ks.b + h * p.ks.h) * KESZ;
  const char* const vp = (const char*)p.v + (b * p.vs.b + h * p.vs.h) * KESZ;
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, (int)((unsigned)(k1 - 1) * krow_b + D * KESZ), 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, (int)((unsigned)(k1 - 1) * vrow_b + D * KESZ), 0x00020000);
  constexpr unsigned NONE = 0x80000000u;  // an offset past any range: zeros

  // The loads of the next tile go out as soon as the registers of this one are read: K's after the scores, V's after
  // the accumulation, so that half a tile of loads is in flight while the wave computes.
  Words<4> kx[2][NK];
  Words<VW> vx[8];
  auto load_k = [&](int key0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = key0 + 16 * u + n;
      const unsigned off = r < k1 ? (unsigned)r * krow_b + 16 * g : NONE;
#pragma unroll
      for (int j = 0; j < NK; ++j) kx[u][j] = load_words<4, AUX>(krs, off + 64 * j);
    }
  };
  auto load_v = [&](int key0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int r = key0 + 16 * (e >> 2) + 4 * g + (e & 3);
      vx[e] = load_words<VW, AUX>(vrs, (r < k1 ? (unsigned)r * vrow_b : NONE) + n * (DL * KESZ));
    }
  };

  f32x4 o[DL], rest[REST ? DL : 1];  // [d][i]: dim DL (4 g + i) + d of row n
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int d = 0; d < DL; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < (REST ? DL : 1); ++d) rest[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int PASS = kWaves * 32;
  const int first = k0 + w * 32;
  if (first < k1) {
    load_k(first);
    load_v(first);
  }
  for (int key0 = first; key0 < k1; key0 += PASS) {
    float s[8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        const Words<4>& k = kx[u][j];
        if constexpr (KV8) {
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            u32x4 y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = MM::widen(k.w[2 * half + i / 2], i & 1);
            acc = MM::run(as_frag<frag>(y), qf[2 * j + half], acc);
          }
        } else {
          acc = MM::run(as_frag<frag>(u32x4{k.w[0], k.w[1], k.w[2], k.w[3]}), qf[j], acc);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) s[4 * u + i] = acc[i] * c;
    }
    if (key0 + PASS < k1) load_k(key0 + PASS);
    if (key0 + 32 > k1) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (key0 + 16 * (e >> 2) + 4 * g + (e & 3) >= k1) s[e] = -INFINITY;
    }
    // The reference maximum moves only when a score has outgrown it by more than 2^slack (flash_fwd.hip).
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, s[e]);
    if (__builtin_amdgcn_ballot_w64(!(mx - m <= W::slack)) != 0) {
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m, mx), alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < DL; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          o[d][i] *= alpha;
          if (REST) rest[REST ? d : 0][i] *= alpha;
        }
    }
    const float ms = m == -INFINITY ? 0.f : m - W::up;
    u32x4 pw[TERMS];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float p0 = __builtin_amdgcn_exp2f(s[2 * i] - ms), p1 = __builtin_amdgcn_exp2f(s[2 * i + 1] - ms);
      l += p0 + p1;
#pragma unroll
      for (int j = 0; j < TERMS; ++j) {
        pw[j][i] = j == 0 ? MP::pack2(W::first(p0), W::first(p1)) : MP::pack2(p0, p1);
        if (j + 1 < TERMS) {
          float y0, y1;
          MP::unpack2(pw[j][i], y0, y1);
          p0 = (p0 - y0) * (j == 0 ? W::later : 1.f);
          p1 = (p1 - y1) * (j == 0 ? W::later : 1.f);
        }
      }
    }
    unsigned y[8][DL / 2];  // [key][pair of dims]
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < DL / 2; ++i) y[e][i] = KV8 ? MMP::widen(vx[e].w[i / 2], i & 1) : vx[e].w[KV8 ? 0 : i];
#pragma unroll
    for (int d = 0; d < DL; ++d) {
      u32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_perm(y[2 * i + 1][d / 2], y[2 * i][d / 2], d & 1 ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int j = TERMS - 1; j >= 0; --j) {
        f32x4& to = REST && j > 0 ? rest[REST ? d : 0] : o[d];
        to = MMP::run(as_frag<pfrag>(v), as_frag<pfrag>(pw[j]), to);
      }
    }
    if (key0 + PASS < k1) load_v(key0 + PASS);
  }

  // the waves' sums: each leaves its rows' O, maximum and sum of weights
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  float* const rec = sm + w * C::REC;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int d0 = 0; d0 < DL; d0 += 4) {
      f32x4 y;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        y[d] = o[d0 + d][i];
        if (REST) {
          const float r = rest[REST ? d0 + d : 0][i] * (1.f / W::later);
          y[d] += fabsf(r) < INFINITY ? r : 0.f;
        }
      }
      *(f32x4*)(rec + n * C::PITCH + DL * (4 * g + i) + d0) = y;
    }
  if (g == 0) {
    rec[16 * C::PITCH + n] = m - W::up;
    rec[16 * C::PITCH + 16 + n] = l;
  }
  __syncthreads();
  const float vmul = KV8 ? p.v_scale[bh] : 1.f;
  for (int t = threadIdx.x; t < nq * (D / 4); t += kWaves * 64) {
    const int i = t / (D / 4), d = t % (D / 4) * 4;
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < kWaves; ++j) mx = fmaxf(mx, sm[j * C::REC + 16 * C::PITCH + i]);
    const float ms = mx == -INFINITY ? 0.f : mx;   // (every score of the chunk -inf: nothing of weight, beside chunks that have some)
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
    float ls = 0.f;
#pragma unroll
    for (int j = 0; j < kWaves; ++j) {
      const float f = __builtin_amdgcn_exp2f(sm[j * C::REC + 16 * C::PITCH + i] - ms);
      ls += sm[j * C::REC + 16 * C::PITCH + 16 + i] * f;
      const f32x4 y = *(const f32x4*)(sm + j * C::REC + i * C::PITCH + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] += y[e] * f;
    }
    const int64_t orow = (int64_t)z * p.Sq + i;
    const float inv = vmul / ls;
    const int64_t at = b * p.os.b + h * p.os.h + orow * p.os.s + d;
    if (p.out32) {
      *(f32x4*)((float*)p.out + at) = a * inv;
    } else {
      const u32x2 st = {M::pack2(a[0] * inv, a[1] * inv), M::pack2(a[2] * inv, a[3] * inv)};
      *(u32x2*)((T*)p.out + at) = st;
    }
    if (d == 0) p.lse[(int64_t)bh * p.lse_bh + orow] = (mx + __builtin_amdgcn_logf(ls)) * 0.6931471805599453f;
  }
}

template <typename T, int D, bool KV8, int TERMS, int W, bool NT>
hipError_t launch_variant(const FwdParams& p, hipStream_t stream) {
  constexpr int smem = DecodeCfg<D, W>::SMEM;
  constexpr auto kernel = rows16_fwd_kernel<T, D, KV8, TERMS, W, NT>;
  const hipError_t e = spa_allow_dynamic_lds<kernel>(smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(p.B * p.H), (unsigned)p.P), dim3(W * 64), smem, stream, p);
  return hipGetLastError();
}

// K and V up to this many bytes stay in the memory-side cache (256 MiB) from one call to the next where a program's other data leave them there; larger ones are
// read past it.  Us a call, three sets of inputs in turn, plain / non-temporal: 16 x 8 heads of 698 keys, D = 128, e4m3 (23 MB) 8.1 / 10.1, bf16 (46) 10.8 /
// 14.5; 32 of 4096, bf16 (67) 15.4 / 16.2; six sets, 32 of 5000, bf16 (82) 20.2 / 18.7; 16 x 32 of 512, bf16 (134) 26.5 / 24.0; 16 x 32 of 4000, e4m3 (524) 91.8 / 83.8.
constexpr int64_t kCachedBytes = (int64_t)64 << 20;
int64_t kv_bytes(const FwdParams& p, int D) {
  const int64_t keys = (int64_t)(p.P - 1) * p.Sk + p.sk_last;
  return (int64_t)p.B * p.H * keys * D * (p.k_scale ? 2 : 4);
}

// Eight waves keep enough loads in flight for 8-bit keys, whose tiles are small; 16-bit ones from memory do with four (32 heads of 32768 keys, bf16,
// D = 128: 82.5 with eight, 80.5 with four).
template <typename T, int D, bool KV8, int TERMS>
hipError_t launch_terms(const FwdParams& p, hipStream_t stream) {
  if (kv_bytes(p, D) <= kCachedBytes) return launch_variant<T, D, KV8, TERMS, 8, false>(p, stream);
  return launch_variant<T, D, KV8, TERMS, KV8 ? 8 : 4, true>(p, stream);
}

template <typename T, int D>
hipError_t launch(const FwdParams& p, hipStream_t stream) {
  const bool exact = p.Sq <= kRowsInFp32;
  if (p.k_scale) return exact ? launch_terms<T, D, true, weight_terms(1)>(p, stream) : launch_terms<T, D, true, weight_terms(16)>(p, stream);
  return exact ? launch_terms<T, D, false, weight_terms(1)>(p, stream) : launch_terms<T, D, false, weight_terms(16)>(p, stream);
}

}  // namespace

// Whether this kernel is the faster one for a call of up to 16 rows (p as for the launch), from 9000 calls of 3 to 4096 heads and 16 to 32768 keys; us a call,
// decode_fwd.hip's kernel (up to three rows) or flash_fwd.hip's / this one.  What it has against it: a workgroup, of eight waves mostly, fills a CU and is long, so
// that a second round of them which is not full, or CUs without one, cost more (`uneven`: long chunks in such a launch), and its start and end count in
// launches of thousands of short ones.
// Rows back to back.  One row: not of 16-bit elements (D = 128: 64 x 32 heads of 48 keys 12.2 / 28.5, 8 of 2048 8.5 / 9.6, 32 of 32768 86.8 / 86.1; D = 64, 8 of
// 700 6.9 / 8.4); of e4m3 ones (D = 64: 64 x 32 heads of 100 keys 22.8 / 14.4, 32 of 4096 12.1 / 10.4, but 5 x 40 of 4096 24.7 / 27.7), at D = 128 in one round
// (32 of 16384 31.9 / 27.9, 2 x 32 of 100 6.8 / 5.5, 64 x 32 of 256 26.3 / 40.2), but for the few workgroups of a call that is not split (8 of 512 7.7 / 7.9, 4 x
// 32 of 16384 106 / 134; of 700 0.95).
// Two rows of 16 bits: 32 of 4096 keys, D = 128 18.3 / 17.2, 8 x 32 of 512, D = 64 11.1 / 9.4; 3 x 32 of 8192 42.5 / 51.3, 16 x 20 of 1024, D = 128
// 32.3 / 38.3, 64 x 32 of 48 14.8 / 28.9; of e4m3 elements 8 x 32 of 2048, D = 128 31.1 / 26.1, but 64 x 32 of 256 35.9 / 40.4.
// Three: 16 x 32 of 1300, D = 128 63.1 / 58.5, e4m3 42.5 / 33.8; 4 x 34 of 8192, in two chunks 130 / 140.
// More: e4m3 elements everywhere (0.41 to 0.9 of flash_fwd.hip's time); 16-bit ones, D = 128, 8 x 32 of 2048 51.3 / 44.0, 20 of 16384, split, 38.3 / 34.2; where
// uneven, up to three quarters of the CUs, 4 x 34 of 2048 33.3 / 37.8.  More than eight rows against a few keys, of which most of the eight waves have none, in
// several rounds: 16 x 32 of 256, D = 128 16.0 / 17.2, 512 x 8 of 48 e4m3 44.9 / 47.4, in between other heads 47.0 / 53.8.
// Rows of other heads in between.  Up to three stay on decode_fwd.hip, which takes neighbouring heads together.  More: e4m3 as back to back, but from memory and not
// split at D = 128 (8 x 32 of 4096 59.4 / 62.4); 16-bit ones as back to back up to what stays in the cache (2 x 32 of 512 keys 11.0 / 10.2; 16 x 20 of 512 20.1 / 26.3).
bool spa_rows16_takes(const FwdParams& p, int D) {
  const bool kv8 = p.k_scale != nullptr, memory = kv_bytes(p, D) > kCachedBytes;
  const int64_t cus = spa_device_cus(), wgs = (int64_t)p.B * p.H * p.P;
  const bool whole = p.P == 1, longer = (int64_t)p.Sk * D >= 2048 * 64, second = wgs > cus && wgs < 2 * cus;
  const bool uneven = longer && (second || (whole && wgs < cus));
  const bool back = p.ks.s == D && p.vs.s == D;
  if (p.Sq > 8 && D == 128 && p.Sk <= 256 && (kv8 ? wgs >= 8 * cus && (!back || p.Sk <= 64) : wgs > cus && wgs < 4 * cus)) return false;
  if (!back) {
    if (p.Sq <= kRowsInFp32) return false;
    if (kv8) return !(D == 128 && memory && whole && p.Sk >= 2048);
    return !memory && !(longer && whole && 4 * wgs < 3 * cus);
  }
  switch (p.Sq) {
    case 1: return kv8 && (D == 64 ? !uneven : wgs <= cus && (!whole || p.Sk <= 256 || 2 * wgs > cus || (2 * wgs == cus && p.Sk < 1024)));
    case 2:
      if (kv8) return D == 64 ? !uneven : !(longer && second) && wgs < 4 * cus;
      return wgs <= cus ? !uneven : wgs >= 2 * cus && p.Sk > 256;
    case 3: return kv8 || !uneven;
    default: return kv8 || !(longer && whole && 4 * wgs < 3 * cus);
  }
}

// As spa_launch_fwd_fewrows, for 1 <= Sq <= 16 rows of calls that are not packed batches.
hipError_t spa_launch_fwd_rows16(const FwdParams& p, int D, int dtype, hipStream_t stream) {
  if (p.causal || p.cu_q || p.q_scale || p.big || p.Sq < 1 || p.Sq > 16 || p.P < 1 || p.P > 65535 || p.Sk < 1 || (int64_t)p.B * p.H > 0x7fffffffLL)
    return hipErrorInvalidValue;
  if (dtype == 1 && D == 128) return launch<__bf16, 128>(p, stream);
  if (dtype == 1 && D == 64) return launch<__bf16, 64>(p, stream);
  if (dtype == 2 && D == 128) return launch<_Float16, 128>(p, stream);
  if (dtype == 2 && D == 64) return launch<_Float16, 64>(p, stream);
  return hipErrorInvalidValue;
}
