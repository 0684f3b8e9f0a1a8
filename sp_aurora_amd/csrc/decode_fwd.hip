// Attention of a handful of query rows over a long K/V (the decode step of a server): the block forward of
// sp_aurora/intel_flash_attn.py:233-296 at Sq <= 3, where the work is reading K and V once.  The MFMA kernels would spend
// a 128-row tile on these rows; here every lane streams 16 bytes of a key row and of a value row per load and the
// scores are plain fused multiply-adds, so that the launch is bound by HBM alone.
//
// Layout of a wave's load: the 64 lanes cover R = 1024 / (D * element size) consecutive key rows, LPR = 64 / R lanes
// a row, lane l holding elements (l % LPR) * E .. + E of row l / LPR (E = 8 for 16-bit, 16 for e4m3 elements).  A
// score is the sum of the LPR lanes' partial dot products (DPP adds inside the 16-lane row); the softmax state
// (running max, running sum, NQ x E accumulators) lives in the group of lanes and covers the rows that group saw.
// At the end the groups of a wave merge by shuffles and the waves of the workgroup through LDS.
//
// Grid: x = batch * head (or group of HP heads), y = key chunk (the key split of the caller: chunk y writes rows y * Sq .. of the result
// tensors it is given).  A packed batch whose keys are cut (chunks of one length, as many as a sequence needs): x = chunk * head, the
// chunks of all sequences numbered through (chunk_of); fp32 partial sums, merged by fewrows_combine_kernel.  256 or 512 threads.
#include "spa_common.h"
#include "spa_host.h"

namespace {

template <int CTRL>
static __device__ __forceinline__ float dpp_add(float x) {
  const int y = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true);
  return x + __builtin_bit_cast(float, y);
}
// Sum over the LPR (4, 8 or 16) consecutive lanes a key row is spread over; every lane of the group gets it.
template <int LPR>
static __device__ __forceinline__ float group_sum(float x) {
  x = dpp_add<0xB1>(x);                   // quad_perm [1,0,3,2]
  x = dpp_add<0x4E>(x);                   // quad_perm [2,3,0,1]
  if (LPR >= 8) x = dpp_add<0x141>(x);    // row_half_mirror: the other quad of the 8 lanes
  if (LPR >= 16) x = dpp_add<0x140>(x);   // row_mirror: the other half of the 16 lanes
  return x;
}

// 16 bytes of a row as floats.
template <typename T, bool KV8>
struct Piece;
template <typename T>
struct Piece<T, false> {
  static constexpr int E = 8;
  static __device__ __forceinline__ void cvt(u32x4 x, float* f) {
#pragma unroll
    for (int j = 0; j < 4; ++j) Mma16<T>::unpack2(x[j], f[2 * j], f[2 * j + 1]);
  }
};
template <typename T>
struct Piece<T, true> {
  static constexpr int E = 16;
  static __device__ __forceinline__ void cvt(u32x4 x, float* f) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)x[j], false);
      const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)x[j], true);
      f[4 * j] = lo[0]; f[4 * j + 1] = lo[1]; f[4 * j + 2] = hi[0]; f[4 * j + 3] = hi[1];
    }
  }
};

typedef float f32x2 __attribute__((ext_vector_type(2)));
// What a chunk of a packed batch leaves in the workspace: per (chunk, head, row) D sums, and behind all of those (max, sum).
__host__ __device__ inline int64_t part_stats(int64_t pairs, int nq, int D) { return pairs * nq * D; }

// The number of a sequence's first chunk of `chunk` keys: those of the sequences before it take no more than this, whatever their lengths
// (rounding each up costs less than one number a sequence), so it needs no sum over them, and the longest sequence decides nothing: all
// numbers are total / chunk + sequences, of which at most one a sequence stays without keys.  (Numbered by sequence, with as many chunks for each as
// twice the mean and the rest in the last, one workgroup a head read most of a cache far longer than the others: one of 32768 tokens and 63 of 512, H = 32,
// D = 128, e4m3 986 -> 106 us, bf16 929 -> 178; one of 16384 and 63 of 1024 487 -> 117, 518 -> 212; four of 8192 and 60 of 1024 262 -> 135, 319 -> 243;
// 64 of 1 to 4 thousand 233 -> 224, 413 -> 415.)
__device__ __forceinline__ int first_chunk(int k_begin, int seq, int chunk) { return (int)((unsigned)k_begin / (unsigned)chunk) + seq; }
// The sequence that owns chunk number `slot`, which of its chunks that is (negative: in front of the first), and its rows.  Called by whole waves: each
// step looks at 64 sequences, evenly spaced; the last reads all offsets at once, so that lists of up to 64 take one memory latency.
struct ChunkOwner {
  int seq, z, q_begin, q_end, k_begin, k_end;
};
__device__ __forceinline__ ChunkOwner chunk_of(const int* cu_q, const int* cu_k, int nseq, int chunk, int slot, int lane) {
  int lo = 0, n = nseq;
  while (n > 64) {
    const int step = (n + 63) / 64, i = lane * step;
    const bool before = i < n && first_chunk(cu_k[lo + i], lo + i, chunk) <= slot;
    const int k = __builtin_popcountll(__builtin_amdgcn_ballot_w64(before));
    if (k > 1) {
      lo += (k - 1) * step;
      n -= (k - 1) * step;
    }
    n = n < step ? n : step;
  }
  const int i = lo + (lane < n ? lane : n - 1);
  const int k0 = cu_k[i], k1 = cu_k[i + 1], q0 = cu_q[i], q1 = cu_q[i + 1];
  const int found = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < n && first_chunk(k0, i, chunk) <= slot)), at = found ? found - 1 : 0;
  ChunkOwner r;
  r.seq = lo + at;
  r.k_begin = __builtin_amdgcn_readlane(k0, at);
  r.k_end = __builtin_amdgcn_readlane(k1, at);
  r.q_begin = __builtin_amdgcn_readlane(q0, at);
  r.q_end = __builtin_amdgcn_readlane(q1, at);
  r.z = slot - first_chunk(r.k_begin, r.seq, chunk);
  return r;
}

// kWaves: waves of a workgroup.  kUnroll: loads of K (and of V) a wave keeps in flight.  NT: the loads carry the non-temporal hint (K and V are read
// once and should not displace anything in the caches).
// HP: neighbouring heads a workgroup takes together, whose pieces of a key row lie side by side.  CHUNKS: a packed batch whose keys are cut (a variant
// of its own: the search costs the others two registers, and with three rows half of the waves).
template <typename T, int D, bool KV8, int NQ, int kUnroll, bool NT, int HP, int kWaves, bool CHUNKS>
__global__ void __launch_bounds__(kWaves * 64) fewrows_fwd_kernel(const FwdParams p) {
  constexpr int AUX = NT ? 2 : 0;
  typedef Piece<T, KV8> Pc;
  constexpr int E = Pc::E;
  constexpr int LPH = D / E;        // lanes per key row and head
  constexpr int LPR = LPH * HP;     // lanes per key row
  constexpr int R = 64 / LPR;       // key rows per load of a wave
  constexpr int KESZ = KV8 ? 1 : 2;
  static_assert((LPH == 4 || LPH == 8 || LPH == 16) && LPR <= 32, "row spread");

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // Workgroups go to the 8 XCDs round robin.  Where a key row of one head is half a cache line (64 e4m3 elements), two
  // neighbouring heads share every line: they are given to workgroups 8 apart, which run on one XCD at about the same
  // time, so that the line comes from HBM once (3.1 -> 4.6-5.1 TB/s; with rows of a whole line or more the same
  // placement is 3-10 % slower than heads round robin).
  // (Chunks of a packed batch, which are not of one size, stay spread over the XCDs: neighbours change places inside 16 workgroups.)
  int bh = blockIdx.x;
  if (D * KESZ * HP < 128) {
    if (!CHUNKS) {
      if ((gridDim.x & 7) == 0) bh = (bh & 7) * (int)(gridDim.x >> 3) + (bh >> 3);
    } else if ((unsigned)(bh | 15) < gridDim.x) {
      bh = (bh & ~15) | ((bh & 7) << 1) | ((bh >> 3) & 1);
    }
  }
  bh *= HP;
  int z = blockIdx.y;
  int b = bh / p.H;
  const int h = bh - b * p.H;                    // the first of the heads
  const int slot = b;                            // (CHUNKS)
  ChunkOwner seq;                                // (packed batches)
  if constexpr (CHUNKS) {
    seq = chunk_of(p.cu_q, p.cu_k, p.B, p.Sk, slot, (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    // (the same in all lanes, which the compiler does not see: descriptors built lane by lane cost up to 15 %)
    for (int* const x : {&seq.q_begin, &seq.q_end, &seq.k_begin, &seq.k_end, &seq.seq, &seq.z}) *x = __builtin_amdgcn_readfirstlane(*x);
    b = seq.seq;
    z = seq.z;
    if (z < 0) return;
    bh = b * p.H + h;
  } else if (p.cu_q) {
    seq = {b, 0, p.cu_q[b], p.cu_q[b + 1], p.cu_k[b], p.cu_k[b + 1]};
  }
  const int c = lane % LPR, g = lane / LPR;
  const int own = c / LPH;                       // this lane's head is h + own
  int k0 = z * p.Sk;
  int k1 = k0 + (z == p.P - 1 && !CHUNKS ? p.sk_last : p.Sk);
  int nq = NQ;                                   // rows of this (batch or sequence, head) that exist
  int64_t q_row0 = 0, k_row0 = 0;                // first row of the sequence in the packed tensors
  int64_t lse_base = (int64_t)bh * p.lse_bh;     // of head h; lse is [B, H, rows], or [H, packed rows] for a packed batch
  if (p.cu_q) {
    // a packed variable-length batch: sequence b owns rows cu_q[b] .. of q / out / lse and cu_k[b] .. of K / V, and
    // this workgroup all of them or chunk z
    q_row0 = seq.q_begin;
    k_row0 = seq.k_begin;
    nq = seq.q_end - seq.q_begin;
    nq = nq < NQ ? nq : NQ;
    k1 = seq.k_end - seq.k_begin;
    if (z > 0 && (int64_t)z * p.Sk >= k1) return;
    if (CHUNKS && k1 - k0 > p.Sk) k1 = k0 + p.Sk;
    lse_base = (int64_t)h * p.lse_bh + q_row0;
    b = 0;
    if (nq <= 0) return;
    if (k1 <= 0) {
      // no keys: the empty sum, out = 0 and lse = -inf
      for (int t = threadIdx.x; t < nq * HP * D; t += kWaves * 64) {
        const int i = t / (HP * D), hd = t / D % HP, d = t % D;
        ((T*)p.out)[(h + hd) * p.os.h + (q_row0 + i) * p.os.s + d] = (T)0.f;
        if (d == 0) p.lse[lse_base + hd * p.lse_bh + i] = -INFINITY;
      }
      return;
    }
  }

  // the rows' queries, this lane's elements, scaled into the exponent's base-2 domain
  const float qmul = (p.negq ? -p.scale_log2 : p.scale_log2) * (KV8 ? p.k_scale[bh + own] : 1.f);
  float qf[NQ][E];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const T* qp = (const T*)p.q + b * p.qs.b + (h + own) * p.qs.h + (q_row0 + (i < nq ? i : nq - 1)) * p.qs.s + c % LPH * E;
#pragma unroll
    for (int e0 = 0; e0 < E; e0 += 8) {
      float t[8];
      Piece<T, false>::cvt(*(const u32x4*)(qp + e0), t);
#pragma unroll
      for (int e = 0; e < 8; ++e) qf[i][e0 + e] = t[e] * qmul;
    }
  }

  // descriptors that end with this chunk's last row: rows past it read as zero and are masked below
  const int64_t krow_b = p.ks.s * KESZ, vrow_b = p.vs.s * KESZ;
  const char* kp = (const char*)p.k + (b * p.ks.b + h * p.ks.h + k_row0 * p.ks.s) * KESZ;
  const char* vp = (const char*)p.v + (b * p.vs.b + h * p.vs.h + k_row0 * p.vs.s) * KESZ;
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, (int)((unsigned)((int64_t)(k1 - 1) * krow_b) + HP * D * KESZ), 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, (int)((unsigned)((int64_t)(k1 - 1) * vrow_b) + HP * D * KESZ), 0x00020000);

  float m[NQ], l[NQ], acc[NQ][E];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    m[i] = -INFINITY;
    l[i] = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) acc[i][e] = 0.f;
  }

  // The loads of the next pass go out as soon as the registers of this pass are read: K's after the scores, V's after
  // the accumulation, so that half a pass of loads is in flight while the wave computes.
  u32x4 kx[kUnroll], vx[kUnroll];
  const unsigned kcol = (unsigned)(g * krow_b) + c * 16, vcol = (unsigned)(g * vrow_b) + c * 16;
  auto load_k = [&](int row0) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      kx[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, (unsigned)((row0 + u * R) * krow_b) + kcol, 0, AUX));
  };
  auto load_v = [&](int row0) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      vx[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vrs, (unsigned)((row0 + u * R) * vrow_b) + vcol, 0, AUX));
  };
  constexpr int kPass = kWaves * kUnroll * R;   // key rows the workgroup takes per pass
  const int first = k0 + wave * (kUnroll * R);
  if (first < k1) {
    load_k(first);
    load_v(first);
  }
  for (int row0 = first; row0 < k1; row0 += kPass) {
    const int row = row0 + g;
    float s[NQ][kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      float kf[E];
      Pc::cvt(kx[u], kf);
      const bool live = row + u * R < k1;
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) d = __builtin_fmaf(qf[i][e], kf[e], d);
        d = group_sum<LPH>(d);
        s[i][u] = live ? d : -INFINITY;
      }
    }
    if (row0 + kPass < k1) load_k(row0 + kPass);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      float mx = m[i];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) mx = fmaxf(mx, s[i][u]);
      // (row0 < k1 for the wave, but this group's rows may all lie past the end: keep the exponents finite)
      const float ms = mx == -INFINITY ? 0.f : mx;
      const float alpha = __builtin_amdgcn_exp2f(m[i] - ms);
      m[i] = mx;
      l[i] *= alpha;
#pragma unroll
      for (int e = 0; e < E; ++e) acc[i][e] *= alpha;
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        s[i][u] = __builtin_amdgcn_exp2f(s[i][u] - ms);
        l[i] += s[i][u];
      }
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      float vf[E];
      Pc::cvt(vx[u], vf);
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[i][e] = __builtin_fmaf(s[i][u], vf[e], acc[i][e]);
    }
    if (row0 + kPass < k1) load_v(row0 + kPass);
  }

  // the R groups of the wave: common max, then sums across the lanes that hold the same elements
  __shared__ float sm_m[NQ][kWaves][HP], sm_l[NQ][kWaves][HP], sm_acc[NQ][kWaves][HP * D];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    float mx = m[i];
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    const float ms = mx == -INFINITY ? 0.f : mx;
    const float w = __builtin_amdgcn_exp2f(m[i] - ms);
    float ls = l[i] * w;
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) ls += __shfl_xor(ls, off, 64);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      float a = acc[i][e] * w;
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) a += __shfl_xor(a, off, 64);
      if (g == 0) sm_acc[i][wave][c * E + e] = a;
    }
    if (g == 0 && c % LPH == 0) {
      sm_m[i][wave][own] = mx;
      sm_l[i][wave][own] = ls;
    }
  }
  __syncthreads();

  // the waves of the workgroup: thread t takes element t % D of one row and head
  for (int t = threadIdx.x; t < NQ * HP * D; t += kWaves * 64) {
    const int i = t / (HP * D), hd = t / D % HP, d = t % D;
    const float vmul = KV8 ? p.v_scale[bh + hd] : 1.f;
    float mx = sm_m[i][0][hd];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, sm_m[i][w][hd]);
    const float ms = mx == -INFINITY ? 0.f : mx;   // (every score of the chunk -inf: nothing of weight, beside chunks that have some)
    float ls = 0.f, a = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float f = __builtin_amdgcn_exp2f(sm_m[i][w][hd] - ms);
      ls += sm_l[i][w][hd] * f;
      a += sm_acc[i][w][hd * D + d] * f;
    }
    if (i >= nq) break;
    if (CHUNKS && seq.k_end - seq.k_begin > p.Sk) {  // not all of the sequence
      const int64_t at = ((int64_t)slot * p.H + h + hd) * NQ + i;
      ((float*)p.part)[at * D + d] = a;
      if (d == 0) *(f32x2*)((float*)p.part + part_stats((int64_t)p.P * p.H, NQ, D) + at * 2) = f32x2{mx, ls};
      continue;
    }
    const int64_t orow = (int64_t)z * p.Sq + i;  // (z = 0 for a sequence of a packed batch)
    T* op = (T*)p.out + b * p.os.b + (h + hd) * p.os.h + (q_row0 + orow) * p.os.s;
    op[d] = (T)(a * vmul / ls);
    if (d == 0) p.lse[lse_base + hd * p.lse_bh + orow] = (mx + __builtin_amdgcn_logf(ls)) * 0.6931471805599453f;
  }
}

// Merges the chunks of a packed batch's rows: a workgroup per (sequence, head), a thread one element of every 256 / D-th chunk, eight of them in flight
// (one after the other they are a chain of memory latencies: 64 caches of 1 to 4 thousand tokens, H = 32, 7.2 -> 6.6 us; 256 chunks of one cache 18 us).
// A sequence of one chunk has its result from the first kernel (1999 caches of 200 tokens and one of 2500, H = 32, 44 -> 15 us).
template <typename T, int D>
__global__ void __launch_bounds__(256) fewrows_combine_kernel(const FwdParams p) {
  constexpr int G = 256 / D, AHEAD = 8;
  const int bh = blockIdx.x, b = bh / p.H, h = bh - b * p.H, tid = threadIdx.x, d = tid % D, g = tid / D;
  const int q_row0 = p.cu_q[b], k_row0 = p.cu_k[b], keys = p.cu_k[b + 1] - k_row0;
  int nq = p.cu_q[b + 1] - q_row0;
  nq = nq < p.Sq ? nq : p.Sq;
  if (keys <= p.Sk) return;  // (written by chunk 0)
  const int first = first_chunk(k_row0, b, p.Sk), have = (keys - 1) / p.Sk + 1, n = have < p.P - first ? have : p.P - first;
  const float vmul = p.k_scale ? p.v_scale[bh] : 1.f;
  __shared__ float weight[256], sums[256], ls[4];
  for (int i = 0; i < nq; ++i) {
    const int64_t at = ((int64_t)first * p.H + h) * p.Sq + i, next = (int64_t)p.H * p.Sq;  // of chunk 0; from chunk to chunk
    const float* const part = (const float*)p.part + at * D + d;
    const f32x2* const ml = (const f32x2*)((const float*)p.part + part_stats((int64_t)p.P * p.H, p.Sq, D)) + at;
    float mx = -INFINITY;  // (every wave for itself)
    for (int j = tid & 63; j < n; j += 64) mx = fmaxf(mx, ml[j * next][0]);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    const float ms = mx == -INFINITY ? 0.f : mx;
    float a = 0.f, l = 0.f;
    for (int j0 = 0; j0 < n; j0 += 256) {
      const int m = n - j0 < 256 ? n - j0 : 256;
      if (tid < m) {
        const f32x2 x = ml[(j0 + tid) * next];
        weight[tid] = __builtin_amdgcn_exp2f(x[0] - ms);
        l += x[1] * weight[tid];
      }
      __syncthreads();
      for (int j = g; j < m; j += AHEAD * G) {
        float x[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) x[u] = part[(j0 + (j + u * G < m ? j + u * G : j)) * next * D];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
          if (j + u * G < m) a += x[u] * weight[j + u * G];
      }
      __syncthreads();
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) l += __shfl_xor(l, off, 64);
    sums[tid] = a;
    if ((tid & 63) == 0) ls[tid >> 6] = l;
    __syncthreads();
    if (g == 0) {
      l = (ls[0] + ls[1]) + (ls[2] + ls[3]);
#pragma unroll
      for (int k = 1; k < G; ++k) a += sums[k * D + d];
      ((T*)p.out)[h * p.os.h + (int64_t)(q_row0 + i) * p.os.s + d] = (T)(a * vmul / l);
      if (d == 0) p.lse[(int64_t)h * p.lse_bh + q_row0 + i] = (mx + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
    }
    __syncthreads();
  }
}

// Loads in flight and the non-temporal hint, measured on twelve decode shapes: four loads beat eight (6-10 %) except with three rows,
// with single heads of 64-byte rows and with 512 bytes of a row; the hint gains 5-15 % on 16-bit K/V, on e4m3 rows of a whole line when the keys are not split, and
// on e4m3 heads taken together (12 % split), and loses where workgroups share lines (64-byte rows) and on split calls of single e4m3 heads.
template <typename T, int D, bool KV8, int NQ, int U, int HP, int W = 4>
hipError_t launch_variant(const FwdParams& p, hipStream_t stream) {
  const bool chunks = p.cu_q && p.part;
  const dim3 grid((unsigned)((int64_t)(chunks ? p.P : p.B) * p.H / HP), chunks ? 1u : (unsigned)p.P), block(W * 64);
  constexpr bool hint = !KV8 || HP > 1;
  if (chunks) {
    hipLaunchKernelGGL((fewrows_fwd_kernel<T, D, KV8, NQ, U, hint, HP, W, true>), grid, block, 0, stream, p);
  } else if (hint || D == 64 || p.P > 1) {
    hipLaunchKernelGGL((fewrows_fwd_kernel<T, D, KV8, NQ, U, hint, HP, W, false>), grid, block, 0, stream, p);
  } else if constexpr (!hint && D != 64) {  // (keys not split)
    hipLaunchKernelGGL((fewrows_fwd_kernel<T, D, KV8, NQ, U, true, HP, W, false>), grid, block, 0, stream, p);
  }
  return hipGetLastError();
}

// A head's piece of a key row is 64 to 256 bytes.  Where neighbouring heads lie side by side (the [rows, H, D] layouts) a workgroup takes
// as many as make 256 bytes: 128-byte requests 4 KiB apart reach 5.1 TB/s, 256-byte ones 6.0 (64 caches of 1 to 4 thousand tokens, H = 32,
// D = 128, e4m3: 256 -> 221 us; fixed length, B = 16, 4096 keys: e4m3 97 -> 85, bf16 D = 64 95 -> 80).  Not where that leaves CUs without
// a workgroup: with one per CU and single heads 44 us, 48 together (B = 1, 32768 keys, e4m3, D = 128).
// Rows of 128 elements, and six workgroups per CU left: as many heads as make 512 bytes, eight loads of them in flight (caches of a quarter to all of
// the length, H = 32, us, 256 bytes with four loads / 512 with four / 512 with eight: 64 of 4096, e4m3 233 / 224 / 217, bf16 416 / 400 / 391; 64 of 8192, e4m3
// - / 411 / 399, bf16 - / 785 / 767; 32 of 4096, e4m3, six workgroups per CU, 112 / 117 / 107; 1 KB with four or eight 234 / 227 for the first).  With
// fewer the last workgroups count for more: 32 caches of 480 to 1915, e4m3, 59.4 / 70.7 / 59.1, 8 of 2 to 8 thousand 65.3 / 61.7 / 66.4.  Two rows, which hold
// half as many waves, gain with 32 heads and lose with 8 (64 of 8192, bf16, 512 with four / eight 204 / 207): four loads, and from eight workgroups per CU on.
// Nor where one sequence, which is twice as long in such a workgroup, is a good part of the whole launch: 255 caches of 256 tokens and one of 2200, e4m3
// 116 -> 155, bf16 194 -> 216.
// A launch that leaves half of the CUs without a workgroup (a caller who did not split the keys) is bound by what its
// few waves keep in flight: eight loads there too.
template <typename T, int D, bool KV8, int NQ>
hipError_t launch_unroll(const FwdParams& p, hipStream_t stream) {
  constexpr int HP = 256 / (D * (KV8 ? 1 : 2));
  const int64_t groups = (int64_t)(p.cu_q && p.part ? 1 : p.B) * p.H * p.P;
  if constexpr (D == 128) {
    constexpr int WIDE = 2 * HP, LOADS = NQ == 2 ? 4 : 8, LEAST = NQ == 1 ? 6 : 8;
    // (a packed batch: what one workgroup has to read, the longest sequence or a chunk, at 44 GB/s; all that is read, at 6 TB/s)
    const double longest = p.Sk * 1024.0 / 44e9, all = (double)p.chunk_rows * p.H * D * (KV8 ? 2 : 4) / 6e12;
    if (p.H % WIDE == 0 && p.ks.h == D && p.vs.h == D && groups / WIDE >= LEAST * spa_device_cus() && (!p.cu_q || 4 * longest <= all))
      return launch_variant<T, D, KV8, NQ, LOADS, WIDE>(p, stream);
  }
  if constexpr (HP > 1) {
    if (p.H % HP == 0 && p.ks.h == D && p.vs.h == D && groups / HP >= spa_device_cus())
      return launch_variant<T, D, KV8, NQ, NQ == 3 ? 8 : 4, HP>(p, stream);
  }
  constexpr int U = NQ == 3 || (KV8 && D == 64) ? 8 : 4;
  // At most one workgroup per CU and chunks of 1 MB of K and V at most: bound by the latency of a wave's passes, which eight waves halve (kernel,
  // us, 4 waves with 8 loads / 8 with 4, bf16, D = 128: 8 heads of 512 keys 8.0 / 7.0, 32 chunks of 2048 23.7 / 20.5, 128 28.5 / 26.0; 256 of 4096 76.8 /
  // 95.1).  e4m3 rows of 128 elements, with twice the sums of a wave to add up, only for few: 8 of 1024 10.2 / 9.2, 64 9.3 / 10.0.
  const int64_t chunk_bytes = (int64_t)p.Sk * D * (KV8 ? 1 : 2) * 2, most = KV8 && D == 128 ? spa_device_cus() / 8 : spa_device_cus();
  if constexpr (NQ < 3)
    if (groups <= most && chunk_bytes <= 1 << 20) return launch_variant<T, D, KV8, NQ, 4, 1, 8>(p, stream);
  if constexpr (U != 8) {
    if (groups * 2 <= spa_device_cus()) return launch_variant<T, D, KV8, NQ, 8, 1>(p, stream);
  }
  return launch_variant<T, D, KV8, NQ, U, 1>(p, stream);
}

template <typename T, int D, bool KV8>
hipError_t launch_nq(const FwdParams& p, hipStream_t stream) {
  switch (p.Sq) {
    case 1: return launch_unroll<T, D, KV8, 1>(p, stream);
    case 2: return launch_unroll<T, D, KV8, 2>(p, stream);
    case 3: return launch_unroll<T, D, KV8, 3>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <typename T, int D>
hipError_t launch_d(const FwdParams& p, hipStream_t stream) {
  const hipError_t e = p.k_scale ? launch_nq<T, D, true>(p, stream) : launch_nq<T, D, false>(p, stream);
  if (e != hipSuccess || !p.cu_q || !p.part) return e;
  hipLaunchKernelGGL((fewrows_combine_kernel<T, D>), dim3((unsigned)(p.B * p.H)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_t(const FwdParams& p, int D, hipStream_t stream) {
  if (D == 128) return launch_d<T, 128>(p, stream);
  if (D == 64) return launch_d<T, 64>(p, stream);
  return hipErrorInvalidValue;
}

}  // namespace

// The caller's FwdParams as for the key-split launch: Sk = keys per chunk, sk_last = keys of the last chunk, P = number of
// chunks; out / lse take rows z * Sq + i of chunk z.  No mask, 1 <= Sq <= 3, 16-bit q / out, K/V of one
// (batch, head) below 2 GiB, 16-byte aligned K/V rows.  A packed variable-length batch: cu_q, cu_k; Sq, Sk = the longest sequence's rows
// and keys, B = sequences, chunk_rows = rows of K and V; with `part` Sk = keys of a chunk and P = spa_fewrows_chunks(), whose sums go there.
hipError_t spa_launch_fwd_fewrows(FwdParams p, int D, int dtype, hipStream_t stream) {
  const bool chunks = p.cu_q && p.part;
  if (p.causal || (p.cu_q && p.P != 1 && !p.part) || p.q_scale || p.big || p.Sq < 1 || p.Sq > 3 || p.P < 1 || p.Sk < 1 ||
      (chunks ? (int64_t)p.P * p.H > 0x7fffffffLL : p.P > 65535))
    return hipErrorInvalidValue;
  if (dtype == 1) return launch_t<__bf16>(p, D, stream);
  if (dtype == 2) return launch_t<_Float16>(p, D, stream);
  return hipErrorInvalidValue;
}

int64_t spa_fewrows_chunks(int nseq, int total_k, int chunk) { return (int64_t)total_k / chunk + nseq; }
int64_t spa_fewrows_part_floats(int64_t pairs, int nq, int D) { return part_stats(pairs, nq, D) + pairs * nq * 2; }
