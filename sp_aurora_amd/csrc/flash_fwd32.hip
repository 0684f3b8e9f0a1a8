// Block attention forward for fp32 tensors: out = softmax(q k^T * scale + mask) v and lse, as in flash_fwd.hip (the same transposed
// formulation; sp_aurora/intel_flash_attn.py:18-126).
//
// Both contractions run on the bf16 matrix instruction.  An fp32 value is the exact sum of three bf16 values, x = h + m + l (8 of
// its 24 significant bits each, rounded to nearest: |m| <= 2^-8 |x|, |l| <= 2^-16 |x|), and a product of two bf16 values is
// exact in fp32.  Of the nine products of two split values the six largest are formed, h h', h m', m h', h l', m m', l h'; the
// three others are less than 2^-23 |x y| together and 2^-26 as a rule, either sign, where the chain of D fused operations that
// they replace rounds D times at 2^-24 of the running sum (the scheme of Henry, Tang and Heinecke, "Leveraging the bfloat16
// artificial intelligence datatype for higher-precision computations", 2019).  Against float64 the results are closer than those of
// v_mfma_f32_32x32x2_f32 were: rms 2.7e-8 and 3.4e-8 at 2048 keys, D = 128, 1.3e-8 and 2.4e-8 at 512, D = 64; with one value per row of q 3.7e-8
// and 4.8e-8, 2.1e-8 and 2.4e-8.
// That instruction does 64 operations a clock and SIMD; six bf16 products at 1024 do 170.
// Bound: the matrix pipe, 6 * 2 * (D / 16) * 32 clocks per 32 x 32 scores, beside 168 vector instructions of softmax and splitting P
// and 30 D / 16 of splitting K and V, once per workgroup and tile.
#include "spa_common.h"
#include "spa_host.h"
#include <math.h>

namespace {

typedef Mma16<__bf16> M;
typedef M::frag frag;

constexpr int F32_BN = 32;        // keys per tile
constexpr int F32_THREADS = 256;  // 4 waves x 32 query rows

// Two values as the three bf16 terms of each, packed in pairs.
__device__ __forceinline__ void split2(float x0, float x1, unsigned& h, unsigned& m, unsigned& l) {
  h = M::pack2(x0, x1);
  const float r0 = x0 - __builtin_bit_cast(float, h << 16), r1 = x1 - __builtin_bit_cast(float, h & 0xffff0000u);
  m = M::pack2(r0, r1);
  l = M::pack2(r0 - __builtin_bit_cast(float, m << 16), r1 - __builtin_bit_cast(float, m & 0xffff0000u));
}
// Eight values as three operands.  They are taken times 2^24: the lowest bit of any fp32 number, denormals included, is then a normal
// bf16 number, where the low terms of values below 2^-110 would be cut off (relative errors of 3e-6 at 1e-35, 3e-3 at 1e-38).  The factors and the
// look at the results cost 5 % at D <= 64 and in the kernel for few rows (causal, us: [1, 4096, 16, 64] 216 -> 228, [1, 512, 32, 128] 38.3 -> 40.5); at
// D = 128 the two accumulators of a score give it back ([1, 4096, 32, 128] 749 -> 741).
constexpr float F32_UP = 0x1p24f, F32_DOWN = 0x1p-48f;  // F32_DOWN: of a product of two
struct Split8 {
  u32x4 h, m, l;
  __device__ __forceinline__ void set(const float* x, float up = F32_UP) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      unsigned a, b, c;
      split2(x[2 * i] * up, x[2 * i + 1] * up, a, b, c);
      h[i] = a;
      m[i] = b;
      l[i] = c;
    }
  }
};
// acc0 + acc1 += a b: the large term alone in acc0, the five small ones in acc1.  Where one product dominates a sum, its h h' is exact in
// acc0 and the sum is rounded once, when the two are added, as a fused operation would round it (with h m' and m h' in acc0 it was
// rounded twice).
__device__ __forceinline__ void mma6(const Split8& a, const Split8& b, f32x16& acc0, f32x16& acc1) {
  const frag ah = as_frag<frag>(a.h), am = as_frag<frag>(a.m), al = as_frag<frag>(a.l);
  const frag bh = as_frag<frag>(b.h), bm = as_frag<frag>(b.m), bl = as_frag<frag>(b.l);
  acc1 = M::run(ah, bl, acc1);
  acc0 = M::run(ah, bh, acc0);
  acc1 = M::run(am, bm, acc1);
  acc1 = M::run(al, bh, acc1);
  acc1 = M::run(ah, bm, acc1);
  acc1 = M::run(am, bh, acc1);
}
template <bool X>
struct Bool {
  static constexpr bool value = X;
};
__device__ __forceinline__ void zero16(f32x16& x) {
#pragma unroll
  for (int v = 0; v < 16; ++v) x[v] = 0.f;
}

// What a wave keeps of its 32 query rows (DV: head dims of its results), and one tile's softmax.
template <int D, int DV = D>
struct Rows {
  Split8 q[D / 16];
  f32x16 o[DV / 32];
  float m_run, l_run, c, down;
  // A score above 2^80 is an infinity in the accumulator, and its row a NaN; one below -2^80 has no weight beside a largest score above
  // -2^70, and rows without one are computed again (lost()).  With a scale that leaves such scores apart the bits that q
  // needs lie higher: below 2^-93 they cannot move an exponent by 2^-50.
  __device__ __forceinline__ void init(const float* row, int hh, bool negate, float scale_log2) {
    start(scale_log2);
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const f32x4* const at = (const f32x4*)(row + ks * 16 + hh * 8);
      split_queries(at[0], at[1], negate, q[ks]);
    }
  }
  __device__ __forceinline__ void split_queries(f32x4 a, f32x4 b, bool negate, Split8& to) const {
    float x[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = negate ? -a[e] : a[e];  // negative softmax scale: -q with |scale|
      x[4 + e] = negate ? -b[e] : b[e];
    }
    to.set(x, c < 0x1p-64f ? 0x1p-40f : F32_UP);
  }
  __device__ __forceinline__ void start(float scale_log2) {
    down = scale_log2 < 0x1p-64f ? 0x1p16f : F32_DOWN;
#pragma unroll
    for (int i = 0; i < DV / 32; ++i) zero16(o[i]);
    m_run = -INFINITY;
    l_run = 0.f;
    c = scale_log2;
  }
  __device__ __forceinline__ bool lost(float m) const { return m < -0x1p70f; }
  // s: raw scores of the tile, keys the row does not see at -inf.  The reference maximum moves only when a row's has grown by
  // more than 2^8 (flash_fwd.hip).
  __device__ __forceinline__ void raise(const f32x16& s) {
    float mx = s[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
    mx = halves_max(mx);
    if (__builtin_amdgcn_ballot_w64(!((mx - m_run) * c <= 8.f)) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2((m_run - m_new) * c);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < DV / 32; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[i][v] *= alpha;
    }
  }
  // -> P as the two operands of the second contraction
  __device__ __forceinline__ void weights(const f32x16& s, Split8 (&pf)[2]) {
    const float mc = m_run == -INFINITY ? 0.f : m_run * c;
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[e] = fast_exp2(__builtin_fmaf(s[8 * u + e], c, -mc));
        ps[e & 1] += x[e];
      }
      pf[u].set(x);
    }
    l_run += ps[0] + ps[1];
  }
};

// Sets the scores of the keys a row does not see to -inf; key0: the tile's first key.
__device__ __forceinline__ void mask_tile(f32x16& s, int key0, int first_row, int qrow, bool causal, int Sk, int hh) {
  if ((causal && key0 + F32_BN - 1 > first_row) || key0 + F32_BN > Sk) {
    const int lim = causal ? (qrow < Sk - 1 ? qrow : Sk - 1) : Sk - 1;
#pragma unroll
    for (int v = 0; v < 16; ++v)
      if (key0 + 8 * (v >> 2) + 4 * hh + (v & 3) > lim) s[v] = -INFINITY;
  }
}

// An infinity (or a value above 2^104) has no three exact terms: the rows that it reaches come out as NaN.  Sums of large values times
// weights above 1 (raise()) overflow where the weighted mean is finite.  Rows with a result that is not finite are computed again here, with the
// fp32 matrix instruction, weights of at most 1 and masked keys left out, so that they are infinite, finite or NaN as the arithmetic of
// the inputs has it: a wave's 32 rows together, over the key tiles it0, it0 + step, ..., until every bad row (bit i: row q0 + i) has met a NaN.
// Bound: that instruction's rate (64 operations a clock and SIMD) and the latency of the loads, which go straight into operands, a tile of V and the next
// of K ahead.  Every row of causal [1, 4096, 32, 128] again, for an infinity in V: 847 -> 2241 us the call, [1, 1024, 16, 64] 33 -> 90 (row by
// row with plain operations [1, 1024, 32, 128] took 8500, now 333); a NaN in K ends the pass where it lies (867 and 89).
// VA: keys of V asked for at a time (16: a tile's, and the next tile's of K, ahead of their use; 4, and of K in parts: where two waves share a SIMD
// and the registers do not hold them).
template <int D, int DV = D, int VA = 16>
struct PlainRows {
  f32x16 o[DV / 32];
  float m, l;  // of row ln, over this lane's keys
  template <typename RowOf>
  __device__ __forceinline__ void run(const FwdParams& p, unsigned bad, int q0, const float* qp, const float* kp, const float* vp, float c, int lane,
                                      int it0, int step, RowOf row_of) {
    const int ln = lane & 31, hh = lane >> 5, qrow = q0 + ln, last = p.Sk - 1;
    const int lim = p.causal && qrow < last ? qrow : last;
    const int kv_end = p.causal && q0 + 32 < p.Sk ? q0 + 32 : p.Sk, nt = (kv_end + F32_BN - 1) / F32_BN;
    // of the products of a score, half hh of the wave takes those of values hh * D / 2 and on
    const auto half_row = [&](const float* base, int64_t stride, int row) { return (const f32x4*)(base + (int64_t)row_of(row) * stride + hh * (D / 2)); };
    f32x4 q[D / 8];
    const f32x4* const qr = half_row(qp, p.qs.s, qrow < p.Sq ? qrow : p.Sq - 1);
#pragma unroll
    for (int i = 0; i < D / 8; ++i) q[i] = p.negq ? -qr[i] : qr[i];
#pragma unroll
    for (int i = 0; i < DV / 32; ++i) zero16(o[i]);
    m = -INFINITY;
    l = 0.f;
    constexpr int KA = VA == 16 ? D / 8 : 4;
    f32x4 k[KA];
    const auto load_keys = [&](int it, int i0) {
      const f32x4* const kr = half_row(kp, p.ks.s, it * F32_BN + ln < p.Sk ? it * F32_BN + ln : last);
#pragma unroll
      for (int i = 0; i < KA; ++i) k[i] = kr[i0 + i];
    };
    if (VA == 16) load_keys(it0, 0);
#pragma unroll 1
    for (int it = it0; it < nt; it += step) {
      const int key0 = it * F32_BN;
      f32x16 s;
      zero16(s);
      const bool whole = !(p.causal && key0 + F32_BN - 1 > q0) && key0 + F32_BN <= p.Sk;  // every row sees every key
      float vx[VA][DV / 32];
      const auto load_values = [&](int v0) {
#pragma unroll
        for (int v = 0; v < VA; ++v) {
          const float* const vr = vp + (int64_t)row_of(key0 + 8 * ((v0 + v) >> 2) + 4 * hh + ((v0 + v) & 3)) * p.vs.s + ln;
#pragma unroll
          for (int i = 0; i < DV / 32; ++i) vx[v][i] = vr[32 * i];
        }
      };
      if (whole && VA == 16) load_values(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < D / 8; ++i) {
        if (VA < 16 && i % KA == 0) {
          __builtin_amdgcn_sched_barrier(0);
          load_keys(it, i);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(k[i % KA][e], q[i][e], s, 0, 0, 0);
      }
      if (VA == 16 && it + step < nt) load_keys(it + step, 0);
      mask_tile(s, key0, q0, qrow, p.causal, p.Sk, hh);
      float mx = s[0];
#pragma unroll
      for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
      const float m_new = fmaxf(m, halves_max(mx)), alpha = m_new == -INFINITY ? 1.f : fast_exp2((m - m_new) * c);
      const float mc = m_new == -INFINITY ? 0.f : m_new * c;
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        s[v] = fast_exp2(__builtin_fmaf(s[v], c, -mc));
        l += s[v];
      }
#pragma unroll
      for (int i = 0; i < DV / 32; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[i][v] *= alpha;
      if (!whole) {
        // a tile with keys that some rows do not see: what lies there (an infinity times a weight of 0) stays out, key by key
        const int n = p.Sk - key0 < F32_BN ? p.Sk - key0 : F32_BN;
#pragma unroll 1
        for (int j = 0; j < n; ++j) {
          const int from = 4 * (j >> 3) + (j & 3);
          float x = s[0];
#pragma unroll
          for (int v = 1; v < 16; ++v) x = from == v ? s[v] : x;
          x = __shfl(x, ln + 32 * ((j >> 2) & 1));
          const float* const vr = vp + (int64_t)row_of(key0 + j) * p.vs.s + 4 * hh;
#pragma unroll
          for (int i = 0; i < DV / 8; ++i) {
            const f32x4 y = *(const f32x4*)(vr + 8 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float sum = __builtin_fmaf(x, y[e], o[i / 4][4 * (i % 4) + e]);
              o[i / 4][4 * (i % 4) + e] = key0 + j <= lim ? sum : o[i / 4][4 * (i % 4) + e];
            }
          }
        }
      } else {
#pragma unroll
        for (int v0 = 0; v0 < 16; v0 += VA) {
          if (VA < 16) load_values(v0);
#pragma unroll
          for (int v = 0; v < VA; ++v)
#pragma unroll
            for (int i = 0; i < DV / 32; ++i) o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(vx[v][i], s[v0 + v], o[i], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      const uint64_t nan = __builtin_amdgcn_ballot_w64(l != l);
      if ((bad & ~(unsigned)(nan | nan >> 32)) == 0) break;
    }
    mfma_settle();
  }
};

// 16-byte chunk permutations of a tile row in LDS, as in flash_fwd.hip.
template <int D>
__device__ __forceinline__ int k_swizzle(int row) {
  constexpr int CPR = D / 8;
  return (row / (16 / CPR)) % CPR;
}
template <int D>
__device__ __forceinline__ int v_swizzle(int row) {
  return D == 128 ? (row & 3) << 2 : D == 64 ? ((row >> 1) & 1) << 2 : 0;
}

template <int D>
struct Fwd32Cfg {
  static constexpr int ROWB = D * 2;               // bytes of a row of one term
  static constexpr int PLANE = F32_BN * ROWB;      // one term of a tile
  static constexpr int TENSOR = 3 * PLANE;
  static constexpr int SMEM = 4 * TENSOR;          // two tiles of K, two of V
  static constexpr int CPR = D / 8;                // 8-value chunks per row
  static constexpr int CHUNKS = F32_BN * CPR;      // of a tile
  static constexpr int NC = (CHUNKS + F32_THREADS - 1) / F32_THREADS;  // per thread
};

// Many rows: a workgroup of 128 query rows; K and V tiles are split once, on their way into LDS, and read by its four waves.
// Causal [1, 4096, 32, 128] 1285 -> 768 us (179 TFLOP/s, 1.07 PFLOP/s of bf16 products), [1, 4096, 16, 64] 446 -> 234, full
// [1, 2048, 16, 32] 119 -> 89.
template <int D>
__global__ void __launch_bounds__(F32_THREADS, D == 128 ? 1 : D == 64 ? 2 : 3) flash_fwd32_kernel(const FwdParams pk) {
  typedef Fwd32Cfg<D> C;
  FwdParams p = pk;  // a variable-length batch rewrites the sizes and bases for its sequence below
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  int b, h, qt;
  if (p.numbered) {
    const int number = blockIdx.x / p.H;
    h = blockIdx.x - number * p.H;
    int nt = 0;
    if (!sequence_tile(p.cu_q, p.B, p.map.P ? p.map.P : 1, 128, number, lane, b, qt, nt)) return;
    qt = nt - 1 - qt;
  } else {
    const int pair = blockIdx.x + blockIdx.z * gridDim.x;
    if (pair >= p.B * p.H) return;
    h = pair % p.H;
    b = pair / p.H;
    qt = p.nqt - 1 - (int)blockIdx.y;
  }
  const int q0 = qt * 128, qw0 = q0 + w * 32;
  if (p.cu_q) {
    const int q_lo = p.cu_q[b], k_lo = p.cu_k[b];
    p.Sq = p.cu_q[b + 1] - q_lo;
    p.Sk = p.cu_k[b + 1] - k_lo;
    p.q = (const float*)p.q + (int64_t)q_lo * p.qs.s;
    p.k = (const float*)p.k + (int64_t)k_lo * p.ks.s;
    p.v = (const float*)p.v + (int64_t)k_lo * p.vs.s;
    p.out = (float*)p.out + (int64_t)q_lo * p.os.s;
    p.lse += q_lo;
    b = 0;
    if (p.Sk <= 0) {
      for (int idx = tid; idx < 128 * (D / 4); idx += F32_THREADS) {
        const int grow = q0 + idx / (D / 4), ch = idx % (D / 4);
        if (grow >= p.Sq) break;
        f32x4 z = {0.f, 0.f, 0.f, 0.f};
        *(f32x4*)((float*)p.out + h * p.os.h + (int64_t)grow * p.os.s + ch * 4) = z;
        if (ch == 0) p.lse[(int64_t)h * p.lse_bh + grow] = -INFINITY;
      }
      return;
    }
  }
  RowMap map = {};
  if (p.map.P) {
    map.init(p.map, p.cu_q ? p.Sq : p.Sq / p.map.P);
    if (p.cu_q) p.Sq = p.Sk = p.Sq * p.map.P;
  }
  if (p.cu_q && q0 >= p.Sq) return;  // a tile of the longest sequence that this one does not have
  auto row_of = [&](int r) { return p.map.P ? map.at(r, p.map.pitch) : r; };        // where row r of the sequence lies
  auto stat_of = [&](int r) { return p.map.P ? map.at(r, p.map.lse_pitch) : r; };   // in lse

  const float* qp = (const float*)p.q + b * p.qs.b + h * p.qs.h;
  const float* kp = (const float*)p.k + b * p.ks.b + h * p.ks.h;
  const float* vp = (const float*)p.v + b * p.vs.b + h * p.vs.h;
  const int qrow = qw0 + ln, qrow_c = qrow < p.Sq ? qrow : p.Sq - 1;
  Rows<D> rows;
  rows.init(qp + (int64_t)row_of(qrow_c) * p.qs.s, hh, p.negq, p.scale_log2);

  const int kv_end = p.causal ? (q0 + 128 < p.Sk ? q0 + 128 : p.Sk) : p.Sk;
  const int nt = (kv_end + F32_BN - 1) / F32_BN;
  const int seen = qw0 / F32_BN + (p.causal ? 1 : nt), ntw = seen < nt ? seen : nt;  // tiles this wave's rows see

  // A thread's 8-value chunks of the tiles after next wait in registers.
  f32x4 kreg[C::NC][2], vreg[C::NC][2];
  auto gload = [&](const float* base, int64_t pitch, int it, f32x4 (&reg)[C::NC][2]) {
#pragma unroll
    for (int i = 0; i < C::NC; ++i) {
      const int ch = tid + i * F32_THREADS;
      if (C::CHUNKS % F32_THREADS == 0 || ch < C::CHUNKS) {
        int r = it * F32_BN + ch / C::CPR;
        r = row_of(r < p.Sk ? r : p.Sk - 1);
        const float* a = base + (int64_t)r * pitch + (ch % C::CPR) * 8;
        reg[i][0] = *(const f32x4*)a;
        reg[i][1] = *(const f32x4*)(a + 4);
      }
    }
  };
  auto lstore = [&](unsigned char* base, bool vt, const f32x4 (&reg)[C::NC][2], int i) {
    {
      const int ch = tid + i * F32_THREADS;
      if (C::CHUNKS % F32_THREADS == 0 || ch < C::CHUNKS) {
        const int r = ch / C::CPR, pos = ch % C::CPR;
        Split8 s;
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = reg[i][e >> 2][e & 3];
        s.set(x);
        unsigned char* const a = base + r * C::ROWB + ((pos ^ (vt ? v_swizzle<D>(r) : k_swizzle<D>(r))) * 16);
        *(u32x4*)a = s.h;
        *(u32x4*)(a + C::PLANE) = s.m;
        *(u32x4*)(a + 2 * C::PLANE) = s.l;
      }
    }
  };
  // LDS: two tiles of K and two of V, K one tile ahead of V
  auto kbuf = [&](int it) { return smem + (it & 1) * C::TENSOR; };
  auto vbuf = [&](int it) { return smem + (2 + (it & 1)) * C::TENSOR; };

  // operand addresses: K rows (16 bytes of row ln), V columns (the transposing read of flash_fwd.hip)
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_u8*)smem;
  unsigned kra[D / 16], vra[D / 32];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) kra[ks] = lds0 + ln * C::ROWB + (((2 * ks + hh) ^ k_swizzle<D>(ln)) * 16);
  {
    const int blk = lane >> 4, e = (lane >> 2) & 3, c4 = lane & 3, krl = 4 * hh + e;
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      const int chunk = db * 4 + (blk & 1) * 2 + (c4 >> 1);
      vra[db] = lds0 + 2 * C::TENSOR + krl * C::ROWB + ((chunk ^ v_swizzle<D>(krl)) * 16) + (c4 & 1) * 8;
    }
  }
  auto v_operand = [&](unsigned a) {
    const u32x2 r0 = lds_read_tr16_b64(a), r1 = lds_read_tr16_b64(a + 8 * C::ROWB);
    u32x4 x;
    x[0] = r0[0];
    x[1] = r0[1];
    x[2] = r1[0];
    x[3] = r1[1];
    return x;
  };
  auto scores = [&](int it, f32x16& s) {
    const unsigned st = (unsigned)((it & 1) * C::TENSOR);
    f32x16 s1;
    zero16(s);
    zero16(s1);
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      Split8 a;
      a.h = lds_read_b128(kra[ks] + st);
      a.m = lds_read_b128(kra[ks] + st + C::PLANE);
      a.l = lds_read_b128(kra[ks] + st + 2 * C::PLANE);
      mma6(a, rows.q[ks], s, s1);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = (s[v] + s1[v]) * rows.down;
  };

  gload(kp, p.ks.s, 0, kreg);
  gload(vp, p.vs.s, 0, vreg);
  f32x4 k1[C::NC][2];
  gload(kp, p.ks.s, 1, k1);
#pragma unroll
  for (int i = 0; i < C::NC; ++i) {
    lstore(kbuf(0), false, kreg, i);
    lstore(vbuf(0), true, vreg, i);
    lstore(kbuf(1), false, k1, i);
  }
  gload(kp, p.ks.s, 2, kreg);
  gload(vp, p.vs.s, 1, vreg);
  __syncthreads();
  f32x16 s;
  scores(0, s);
  mfma_settle();
  __syncthreads();
  // Step `it`: the weights of tile `it` are formed while the scores of tile it + 1 are, and the tiles after next are split and
  // written while the products with V run: one wave on a SIMD keeps the matrix pipe and the vector unit busy together.  The
  // compiler is told the mixture, since it would put the two streams one after the other; LDS writes come
  // after the reads of the same quarter in program order, past which they could not be moved.
  constexpr int CH = D > 32 ? 2 : 1;              // head-dim blocks at a time: chains of dependent matrix instructions
  constexpr int GROUPS = 2 * (D / 32) / CH;       // of products with V
  auto v_group = [&](unsigned st, int g, Split8 (&a)[CH]) {
    const int u = g / (GROUPS / 2), db = g % (GROUPS / 2) * CH;
#pragma unroll
    for (int x = 0; x < CH; ++x) {
      const unsigned at = vra[db + x] + st + u * 16 * C::ROWB;
      a[x].h = v_operand(at);
      a[x].m = v_operand(at + C::PLANE);
      a[x].l = v_operand(at + 2 * C::PLANE);
    }
  };
  auto store_next = [&](int it, int i) {  // quarter i of what a thread writes: half of K, or of V (all of each at D <= 64)
    if (i < C::NC)
      lstore(kbuf(it), false, kreg, i);
    else if (i < 2 * C::NC)
      lstore(vbuf(it + 1), true, vreg, i - C::NC);
  };
  auto step = [&](int it, auto last_c) {
    constexpr bool last = decltype(last_c)::value;
    const unsigned st = (unsigned)((it & 1) * C::TENSOR);
    mask_tile(s, it * F32_BN, qw0, qrow, p.causal, p.Sk, hh);
    rows.raise(s);
    f32x16 sn;
    Split8 pf[2];
    __builtin_amdgcn_sched_barrier(0);
    if (!last) scores(it + 1, sn);
    rows.weights(s, pf);
    Split8 a[2][CH];
    v_group(st, 0, a[0]);
    if (!last) {
#pragma unroll
      for (int i = 0; i < 6 * (D / 16); ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, (192 + 6 * (D / 16) - 1) / (6 * (D / 16)), 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      const int u = g / (GROUPS / 2), db = g % (GROUPS / 2) * CH;
      if (g + 1 < GROUPS) v_group(st, g + 1, a[(g + 1) & 1]);
#pragma unroll
      for (int term = 0; term < 6; ++term)
#pragma unroll
        for (int x = 0; x < CH; ++x) {
          const Split8& av = a[g & 1][x];
          const frag va = as_frag<frag>(term == 2 || term == 3 ? av.m : term == 4 ? av.l : av.h);
          const frag pb = as_frag<frag>(term == 0 ? pf[u].l : term == 1 || term == 2 ? pf[u].m : pf[u].h);
          rows.o[db + x] = M::run(va, pb, rows.o[db + x]);
        }
      store_next(it, g);
#pragma unroll
      for (int i = 0; i < 6 * CH; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, D > 32 ? 4 : 8, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    gload(kp, p.ks.s, it + 3, kreg);
    gload(vp, p.vs.s, it + 2, vreg);
    if (!last) s = sn;
  };
  int it = 0;
  for (; it + 1 < ntw; ++it) {
    step(it, Bool<false>());
    __syncthreads();
  }
  step(it, Bool<true>());
  while (++it < nt) {  // the workgroup's later rows see more
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * C::NC; ++i) store_next(it, i);
    gload(kp, p.ks.s, it + 3, kreg);
    gload(vp, p.vs.s, it + 2, vreg);
  }

  float* const obase = (float*)p.out + b * p.os.b + h * p.os.h;
  float* const lbase = p.lse + ((int64_t)b * p.H + h) * p.lse_bh;
  bool bad = false;
  auto store = [&](const f32x16 (&o)[D / 32], float m, float l, float down) {
    float* op = obase + (int64_t)row_of(qrow) * p.os.s;
    const float inv = 1.f / l * down;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 st;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          st[e] = o[db][4 * g + e] * inv;
          bad |= !(fabsf(st[e]) < INFINITY);
        }
        *(f32x4*)(op + db * 32 + 8 * g + 4 * hh) = st;
      }
    if (hh == 0) lbase[stat_of(qrow)] = (m * rows.c + fast_log2(l)) * 0.6931471805599453f;
  };
  const float l_tot = halves_sum(rows.l_run);
  if (qrow < p.Sq) {
    store(rows.o, rows.m_run, l_tot, F32_DOWN);
    bad |= rows.lost(rows.m_run);
  }
  const uint64_t again = __builtin_amdgcn_ballot_w64(bad);
  if (again) {
    const unsigned which = (unsigned)(again | again >> 32);
    PlainRows<D> plain;
    plain.run(p, which, qw0, qp, kp, vp, rows.c, lane, 0, 1, row_of);
    const float l = halves_sum(plain.l);
    if (which >> ln & 1) store(plain.o, plain.m, l, 1.f);
  }
}

// Few rows: a launch of the kernel above with fewer workgroups than CUs lasts as long as one wave's chain over all key tiles.
// Here a workgroup owns 32 query rows and its NW waves take every NW-th key tile, without a barrier in the loop: a tile of K goes
// straight to LDS that is the wave's own (whole rows at a time; read by the lanes that need them, 16 bytes of 32 rows are 32 cache lines
// an instruction), V straight into operands (a column of V 32 lanes wide per key).  The rows' own three terms are formed once and lie in LDS.
// The waves' (O, m, l) are combined through LDS at the end.  Where that leaves CUs without a workgroup, D / DV of them take the same rows and keys, each
// for its DV head dims of the result: the scores are formed again, the splitting of V, its products and the combination are shared out.
// Bound: the vector instructions that split K and V (D = 128: 830 of 1000 a tile and wave, 4000 clocks beside 3072 of the matrix pipe), with two
// waves a SIMD to run beside each other.  Before, K came as operands row by row, a branch for rows in shards stood around every load, D = 128 had one wave a SIMD,
// and half of the CUs were idle under small grids: [1, 8, 512, 64] 14.6 -> 10.9 us, [1, 8, 512, 128] 28.5 -> 17.5 (with whole rows 21), [1, 8, 256, 128]
// 17.1 -> 9.8, [1, 12, 2048, 128] causal 177 -> 115.
template <int D, int DV, int NW>
struct Fwd32SplitCfg {
  static constexpr int REC = 64 * (DV / 8) * 4;              // floats of one wave's O
  static constexpr int QPLANE = 32 * D * 2;                  // one term of the rows
  static constexpr int KTILE = F32_BN * D * 4;
  static constexpr int CPR = D / 4;                          // 16-byte chunks of a row of K
  static constexpr int LOOP = 3 * QPLANE + NW * KTILE, COMBINE = (NW * (REC + 128) + NW) * 4;
  static constexpr int SMEM = LOOP > COMBINE ? LOOP : COMBINE;
  // chunk permutation of a row: 16 rows at one chunk lie in 16 different 16-byte bank groups
  static __device__ __forceinline__ int swizzle(int row) { return D == 32 ? row >> 1 & 7 : row & 15; }
};

template <int D, int DV, int NW, bool MAP>
__global__ void __launch_bounds__(64 * NW, 1) flash_fwd32_splitk_kernel(const FwdParams p) {
  typedef Fwd32SplitCfg<D, DV, NW> C;
  constexpr int PARTS = D / DV;
  extern __shared__ __align__(16) unsigned char smem[];
  float* const sm = (float*)smem;
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pair = blockIdx.x + blockIdx.z * gridDim.x;
  if (pair >= p.B * p.H) return;
  const int h = pair % p.H, b = pair / p.H;
  const int q0 = (p.nqt - 1 - (int)blockIdx.y / PARTS) * 32, d0 = (int)blockIdx.y % PARTS * DV;
  RowMap map = {};
  if (MAP) map.init(p.map, p.Sq / p.map.P);
  auto row_of = [&](int r) { return MAP ? map.at(r, p.map.pitch) : r; };        // where row r of the sequence lies
  auto stat_of = [&](int r) { return MAP ? map.at(r, p.map.lse_pitch) : r; };   // in lse
  const float* qp = (const float*)p.q + b * p.qs.b + h * p.qs.h;
  const float* kp = (const float*)p.k + b * p.ks.b + h * p.ks.h;
  const float* vp = (const float*)p.v + b * p.vs.b + h * p.vs.h + d0;
  const int qrow = q0 + ln;
  const int kv_end = p.causal ? (q0 + 32 < p.Sk ? q0 + 32 : p.Sk) : p.Sk;
  const int nt = (kv_end + F32_BN - 1) / F32_BN;

  const unsigned lds0 = (unsigned)(uintptr_t)(lds_u8*)smem, ktile = lds0 + 3 * C::QPLANE + w * C::KTILE;
  auto load_keys = [&](int it) {  // (rows past the end: the last one, masked below)
#pragma unroll
    for (int j = 0; j < C::KTILE / 1024; ++j) {
      const int slot = j * 64 + lane, row = slot / C::CPR, r = it * F32_BN + row;
      const float* a = kp + (int64_t)row_of(r < p.Sk ? r : p.Sk - 1) * p.ks.s + ((slot % C::CPR) ^ C::swizzle(row)) * 4;
      load_to_lds_b128(a, ktile + j * 1024);
    }
  };
  float vx[2][DV / 32][8];
  auto load_values = [&](int it) {
    // operand element e of half u: key 16 u + 8 (e / 4) + 4 hh + e % 4, as the rows of an accumulator lie
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int r = it * F32_BN + 16 * u + 8 * (e >> 2) + 4 * hh + (e & 3);
        const float* v = vp + (int64_t)row_of(r < p.Sk ? r : p.Sk - 1) * p.vs.s + ln;
#pragma unroll
        for (int db = 0; db < DV / 32; ++db) vx[u][db][e] = v[db * 32];
      }
  };
  constexpr int CH = DV == 64 ? 2 : 1;  // head-dim blocks at a time (of four only one, so that the registers hold both halves of a tile's keys)
  Rows<D, DV> rows;
  rows.start(p.scale_log2);
  // (a whole chunk of eight values a thread, or none)
  const int qr = tid / (D / 8), qc = tid % (D / 8);
  static_assert(32 * D / 8 <= 64 * NW, "the rows' chunks are split in one go");
  f32x4 qa, qb;
  if (qr < 32) {
    const int r = q0 + qr < p.Sq ? q0 + qr : p.Sq - 1;
    const f32x4* const at = (const f32x4*)(qp + (int64_t)row_of(r) * p.qs.s + qc * 8);
    qa = at[0];
    qb = at[1];
  }
  __builtin_amdgcn_sched_barrier(0);
  if (w < nt) {
    load_keys(w);
    load_values(w);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (qr < 32) {
    Split8 x;
    rows.split_queries(qa, qb, p.negq, x);
    unsigned char* const to = smem + qr * (D * 2) + (qc ^ k_swizzle<D>(qr)) * 16;
    *(u32x4*)to = x.h;
    *(u32x4*)(to + C::QPLANE) = x.m;
    *(u32x4*)(to + 2 * C::QPLANE) = x.l;
  }
  __syncthreads();
  for (int it = w; it < nt; it += NW) {
    const int key0 = it * F32_BN;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tile of K (and of V, which was asked for with it)
    f32x16 s, s1;
    zero16(s);
    zero16(s1);
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      float x[8];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const f32x4 y = __builtin_bit_cast(f32x4, lds_read_b128(ktile + ln * (D * 4) + ((4 * ks + 2 * hh + j) ^ C::swizzle(ln)) * 16));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * j + e] = y[e];
      }
      Split8 a, q;
      a.set(x);
      const unsigned at = lds0 + ln * (D * 2) + ((2 * ks + hh) ^ k_swizzle<D>(ln)) * 16;
      q.h = lds_read_b128(at);
      q.m = lds_read_b128(at + C::QPLANE);
      q.l = lds_read_b128(at + 2 * C::QPLANE);
      mma6(a, q, s, s1);
    }
    if (it + NW < nt) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this tile of K has been read
      load_keys(it + NW);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = (s[v] + s1[v]) * rows.down;
    mask_tile(s, key0, q0, qrow, p.causal, p.Sk, hh);
    Split8 pf[2];
    rows.raise(s);
    rows.weights(s, pf);
    // (the small terms of all of the tile's keys first: 5 to 8 % less rounding error)
#pragma unroll
    for (int db = 0; db < DV / 32; db += CH) {
      Split8 va[2][CH];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int x = 0; x < CH; ++x) va[u][x].set(vx[u][db + x]);
#pragma unroll
      for (int term = 0; term < 6; ++term)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int x = 0; x < CH; ++x) {
            const Split8 &vs = va[u][x], &ps = pf[u];
            const frag a = as_frag<frag>(term == 2 || term == 3 ? vs.m : term == 4 ? vs.l : vs.h);
            const frag pb = as_frag<frag>(term == 0 ? ps.l : term == 1 || term == 2 ? ps.m : ps.h);
            rows.o[db + x] = M::run(a, pb, rows.o[db + x]);
          }
    }
    if (it + NW < nt) load_values(it + NW);
  }
  __syncthreads();  // (the same LDS again)
  // ---- combine: every wave leaves its unscaled O (lane-private order) and (m, l); wave j then finishes the
  // 16-byte pieces j, j + NW, ... of every row (of `which`) ----
  constexpr int NPC = DV / 8;  // 16-byte pieces per lane: (db, g)
  float* const obase = (float*)p.out + b * p.os.b + h * p.os.h + d0;
  float* const lbase = p.lse + ((int64_t)b * p.H + h) * p.lse_bh;
  bool bad = false;
  auto combine = [&](const f32x16 (&o)[DV / 32], float m, float l, float down, unsigned which) {
    float* const orec = sm + w * (C::REC + 128);
#pragma unroll
    for (int db = 0; db < DV / 32; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 st;
#pragma unroll
        for (int e = 0; e < 4; ++e) st[e] = o[db][4 * g + e];
        *(f32x4*)(orec + ((db * 4 + g) * 64 + lane) * 4) = st;
      }
    if (hh == 0) {
      orec[C::REC + ln] = m;
      orec[C::REC + 32 + ln] = l;
    }
    __syncthreads();
    float mw[NW], m_all = -INFINITY;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      mw[j] = sm[j * (C::REC + 128) + C::REC + ln];
      m_all = fmaxf(m_all, mw[j]);
    }
    float aw[NW], l_all = 0.f;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      aw[j] = mw[j] == -INFINITY ? 0.f : fast_exp2((mw[j] - m_all) * rows.c);  // a wave without a visible key
      l_all += aw[j] * sm[j * (C::REC + 128) + C::REC + 32 + ln];
    }
    const float inv = 1.f / l_all * down;
    if (qrow < p.Sq && (which >> ln & 1)) {
      bad = rows.lost(m_all);
      float* const op = obase + (int64_t)row_of(qrow) * p.os.s;
      for (int pc = w; pc < NPC; pc += NW) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NW; ++j) {
          const f32x4 x = *(const f32x4*)(sm + j * (C::REC + 128) + (pc * 64 + lane) * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e] += aw[j] * x[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[e] *= inv;
          bad |= !(fabsf(acc[e]) < INFINITY);
        }
        *(f32x4*)(op + (pc / 4) * 32 + 8 * (pc % 4) + 4 * hh) = acc;
      }
      if (w == 0 && hh == 0 && d0 == 0) lbase[stat_of(qrow)] = (m_all * rows.c + fast_log2(l_all)) * 0.6931471805599453f;
    }
  };
  combine(rows.o, rows.m_run, halves_sum(rows.l_run), F32_DOWN, ~0u);
  const uint64_t again = __builtin_amdgcn_ballot_w64(bad);
  unsigned* const flags = (unsigned*)(sm + NW * (C::REC + 128));
  if (lane == 0) flags[w] = (unsigned)(again | again >> 32);
  __syncthreads();
  unsigned which = 0;
#pragma unroll
  for (int j = 0; j < NW; ++j) which |= flags[j];
  if (__builtin_amdgcn_readfirstlane(which)) {
    constexpr int VA = D == 128 && DV >= 64 ? 4 : 16;
    PlainRows<D, DV, VA> plain;
    plain.run(p, which, q0, qp, kp, vp, rows.c, lane, w, NW, row_of);
    combine(plain.o, plain.m, halves_sum(plain.l), 1.f, which);
  }
}

// parts: workgroups that share the rows of a tile
template <auto kernel>
hipError_t launch(int threads, int smem, int rows, int parts, FwdParams p, hipStream_t stream) {
  const hipError_t e = spa_allow_dynamic_lds<kernel>(smem);
  if (e != hipSuccess) return e;
  dim3 grid;
  if (p.cu_q) {
    if (!spa_varlen_grid(p.H, p.B, p.lse_bh, p.Sq, rows, 1, grid, p.numbered)) return hipErrorInvalidValue;
  } else {
    if (p.nqt * parts > 65535) return hipErrorInvalidValue;
    grid = spa_head_groups((int64_t)p.B * p.H, p.nqt * parts);
  }
  hipLaunchKernelGGL(kernel, grid, dim3(threads), smem, stream, p);
  return hipGetLastError();
}

// (rows in shards are looked up row by row: a variant of its own, since the branch would stand around every load)
template <int D, int DV>
hipError_t launch_part(const FwdParams& p, hipStream_t stream) {
  constexpr int NW = 8, smem = Fwd32SplitCfg<D, DV, NW>::SMEM, parts = D / DV;
  return p.map.P ? launch<flash_fwd32_splitk_kernel<D, DV, NW, true>>(64 * NW, smem, 32, parts, p, stream)
                 : launch<flash_fwd32_splitk_kernel<D, DV, NW, false>>(64 * NW, smem, 32, parts, p, stream);
}
template <int D>
hipError_t launch_splitk(const FwdParams& p, hipStream_t stream) {
  const int64_t tiles = (int64_t)p.B * p.H * p.nqt;
  // as many as there are CUs for: 128 tiles of 512 keys at D = 64 in one, two parts 12.4, 10.9 us, D = 128 21.2, 17.4; 64 of 256 keys at D = 128 in
  // one, two, four 12.8, 10.2, 9.5; with more workgroups than CUs a second round costs more: 200 tiles of 777 keys 31 and 37
  int parts = 1;
  while (parts * 2 * tiles <= spa_device_cus()) parts *= 2;
  if constexpr (D == 128)
    if (parts >= 4) return launch_part<D, D / 4>(p, stream);
  if constexpr (D >= 64)
    if (parts >= 2) return launch_part<D, D / 2>(p, stream);
  return launch_part<D, D>(p, stream);
}

#ifdef SPA_FWD32_WIDE_UNIT
}  // namespace
hipError_t spa_launch_fwd32_shared_keys_128(const FwdParams& p, hipStream_t stream) { return launch_splitk<128>(p, stream); }
#else
// Whether the waves of a workgroup share out the keys of 32 rows rather than taking 32 rows each.  Microseconds of a launch, less what both have in common, from
// 5700 launches of 1 to 4000 rows and keys and 1 to 512 heads (of which the kernel that is taken is more than 5 % the slower one for 54, 2 us at most): workgroups of the
// kernel for many rows begin `begin` later, take the tiles of the longest chain at `first` each alone on their CU and at `full` each and workgroup where
// several share it, and each round of them `round`; those for few rows, one to a CU, `start` and `step` for every eighth tile.  Not causal, whole rounds of
// workgroups; causal, heaviest first, the longest or all of them over the CUs.  (Short calls, many / few rows: 16 heads of 14 causal rows, D = 32 9.9 / 6.8 us; 4 x 16 of
// 20, D = 128 17.8 / 8.9; 4 x 8 of 409 against 3565, D = 128 307 / 228, of 2964 against 1299 413 / 550.)
bool keys_shared(const FwdParams& p, int D) {
  const double first = D == 128 ? 2.1 : D == 64 ? 1.53 : 1.49, full = D == 128 ? 2.11 : 1.04;
  const double begin = D == 128 ? 3.2 : D == 64 ? 2.7 : 2.0, round = D == 128 ? 1.9 : D == 64 ? 0.55 : 0.7;
  const double start = D == 128 ? 4.45 : D == 64 ? 3.55 : 2.85, step = D == 128 ? 5.52 : D == 64 ? 3.9 : 2.94;
  const double r = (p.Sq + 31) / 32, k = (p.Sk + F32_BN - 1) / F32_BN, cus = spa_device_cus(), pairs = (double)p.B * p.H;
  const double chain = p.causal && r < k ? r : k;
  // tiles that 32 rows see, and 128
  const double seen = !p.causal ? k : r <= k ? (r + 1) / 2 : k - k * (k - 1) / (2 * r), seen4 = seen + 1.5 < k ? seen + 1.5 : k;
  const double few = pairs * r / cus, many = pairs * ((p.Sq + 127) / 128) / cus;
  double t_few, t_many;
  if (p.causal) {
    const double longest = start + chain / 8 * step, all = few * (start + seen / 8 * step);
    t_few = longest > all ? longest : all;
    const double work = many * (seen4 * full + round);
    t_many = begin + (chain * first > work ? chain * first : work);
  } else {
    t_few = ceil(few) * (start + k / 8 * step);
    t_many = begin + (many <= 1 ? k * first : ceil(many) * (k * full + round));
  }
  return t_few < t_many;
}

}  // namespace

hipError_t spa_launch_fwd32_shared_keys_128(const FwdParams& p, hipStream_t stream);

// One block pair, or whole sequences in shards (p.map).  Returns hipSuccess, or hipErrorInvalidValue for an unsupported D.
hipError_t spa_launch_fwd32(FwdParams p, int D, hipStream_t stream) {
  if (p.epi != SPA_EPI_PLAIN || p.P != 1 || p.nranks != 1) return hipErrorInvalidValue;  // ring steps merge with the separate kernel
  const int knob = spa_knob(SPA_KNOB_FWD32_SPLIT);
  if (!p.cu_q && knob != 1 && (knob == 2 || keys_shared(p, D))) {
    p.nqt = (p.Sq + 31) / 32;
    if (D == 128) return spa_launch_fwd32_shared_keys_128(p, stream);
    if (D == 64) return launch_splitk<64>(p, stream);
    if (D == 32) return launch_splitk<32>(p, stream);
    return hipErrorInvalidValue;
  }
  p.nqt = (p.Sq + 127) / 128;
  if (D == 128) return launch<flash_fwd32_kernel<128>>(F32_THREADS, Fwd32Cfg<128>::SMEM, 128, 1, p, stream);
  if (D == 64) return launch<flash_fwd32_kernel<64>>(F32_THREADS, Fwd32Cfg<64>::SMEM, 128, 1, p, stream);
  if (D == 32) return launch<flash_fwd32_kernel<32>>(F32_THREADS, Fwd32Cfg<32>::SMEM, 128, 1, p, stream);
  return hipErrorInvalidValue;
}
#endif
