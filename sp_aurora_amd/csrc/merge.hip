// Ring-step merge and final cast: plain coalesced HBM streams.
//   merge    : (out_acc, lse_acc) <- logaddexp-combine with one block's (out, lse)
//              stands in for update_out_and_lse (sp_aurora/utils.py:47-147)
//   finalize : out = cast(out_acc)   (sp_aurora/intel_ring_flash_attn.py:141-143)
//   delta    : delta = rowsum(dout * out), first pass of the block-wise backward
// One thread owns 8 head dims of a (b, h, s) row (all loads are issued before the first store); the D/8 threads of a row
// sit in one wavefront, so every lane of the row has read lse_acc before the row's first lane overwrites it.  32-bit row
// arithmetic, the batch index comes from the grid.
#include "spa_common.h"

namespace {

struct RowIdx {
  int b, h, s;
};

// Rows of one batch entry are enumerated with the head index fastest after the sequence index of
// the [B,S,H,D] accumulator: row = s*H + h (32-bit: a batch entry holds fewer than 2^31 rows, the
// launchers check it); the batch index is the grid's y dimension.
static __device__ __forceinline__ RowIdx decode_row(unsigned row, int H) {
  RowIdx r;
  r.s = (int)(row / (unsigned)H);
  r.h = (int)(row - (unsigned)r.s * (unsigned)H);
  r.b = (int)blockIdx.y;
  return r;
}

constexpr int ROWS_PER_THREAD = 1;  // rows a thread takes (two, `half` rows apart with all loads first, measured 10 % slower on the merge)

template <typename T>
struct Load8;  // 8 consecutive elements as floats

template <>
struct Load8<float> {
  static __device__ __forceinline__ void ld(const float* p, float* x) {
    const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 4);
    x[0] = a[0]; x[1] = a[1]; x[2] = a[2]; x[3] = a[3];
    x[4] = b[0]; x[5] = b[1]; x[6] = b[2]; x[7] = b[3];
  }
  static __device__ __forceinline__ void st(float* p, const float* x) {
    f32x4 a, b;
    a[0] = x[0]; a[1] = x[1]; a[2] = x[2]; a[3] = x[3];
    b[0] = x[4]; b[1] = x[5]; b[2] = x[6]; b[3] = x[7];
    *(f32x4*)p = a;
    *(f32x4*)(p + 4) = b;
  }
};

template <>
struct Load8<__bf16> {
  static __device__ __forceinline__ void ld(const __bf16* p, float* x) {
    const u32x4 a = *(const u32x4*)p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __builtin_bit_cast(float, a[i] << 16);
      x[2 * i + 1] = __builtin_bit_cast(float, a[i] & 0xffff0000u);
    }
  }
  static __device__ __forceinline__ void st(__bf16* p, const float* x) {
    u32x4 a;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = Mma16<__bf16>::pack2(x[2 * i], x[2 * i + 1]);
    *(u32x4*)p = a;
  }
};

template <>
struct Load8<_Float16> {
  static __device__ __forceinline__ void ld(const _Float16* p, float* x) {
    const f16x8 a = *(const f16x8*)p;
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = (float)a[i];
  }
  static __device__ __forceinline__ void st(_Float16* p, const float* x) {
    u32x4 a;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = Mma16<_Float16>::pack2(x[2 * i], x[2 * i + 1]);
    *(u32x4*)p = a;
  }
};

// merge: a thread owns 4 dims of either half of a row, 4 ch .. and D / 2 + 4 ch .., so that the lanes' 16 bytes of the fp32 sums lie back to back (8
// consecutive dims a thread: two accesses of every other 16 bytes).  A workgroup takes consecutive rows of one head (by_head): its lse is one
// piece of memory, where rows of 16 heads, heads fastest, read and wrote 4 bytes of 16 cache lines each, lines that 31 other workgroups
// on all XCDs wrote into as well.  Bound: the memory-side cache and HBM.  32 heads of 1024 rows, D = 128, bf16 (42 MB): 9.1 us, the
// dims split 8.3, rows by head 8.0 (5.3 TB/s); 2 x 32 of 2048 29.2 -> 26.5 us; D = 64 5.4 -> 4.9.
template <typename T>
__device__ __forceinline__ void load44(const T* p, int half, float* x);
template <>
__device__ __forceinline__ void load44<float>(const float* p, int half, float* x) {
  const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + half);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = a[i];
    x[4 + i] = b[i];
  }
}
template <>
__device__ __forceinline__ void load44<__bf16>(const __bf16* p, int half, float* x) {
  const u32x2 a = *(const u32x2*)p, b = *(const u32x2*)(p + half);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    x[2 * i] = __builtin_bit_cast(float, a[i] << 16);
    x[2 * i + 1] = __builtin_bit_cast(float, a[i] & 0xffff0000u);
    x[4 + 2 * i] = __builtin_bit_cast(float, b[i] << 16);
    x[4 + 2 * i + 1] = __builtin_bit_cast(float, b[i] & 0xffff0000u);
  }
}
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
template <>
__device__ __forceinline__ void load44<_Float16>(const _Float16* p, int half, float* x) {
  const f16x4 a = *(const f16x4*)p, b = *(const f16x4*)(p + half);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = (float)a[i];
    x[4 + i] = (float)b[i];
  }
}

template <typename T, bool INIT>
__global__ void __launch_bounds__(256) merge_kernel(float* __restrict__ out_acc, float* __restrict__ lse_acc,
                                                    const T* __restrict__ blk_out,
                                                    const float* __restrict__ blk_lse, int H, int Sq,
                                                    int cpr_shift /* log2(D/8) */, bool by_head, Strides3 as, Strides3 bs, int64_t acc_lse_bh) {
  const int ch = (int)(threadIdx.x & ((1u << cpr_shift) - 1u)), half = 4 << cpr_shift;
  RowIdx r;
  if (by_head) {
    const unsigned block = blockIdx.x / (unsigned)H;
    r.h = (int)(blockIdx.x - block * (unsigned)H);
    r.s = (int)((block * 256u + threadIdx.x) >> cpr_shift);
    r.b = (int)blockIdx.y;
  } else {
    r = decode_row((blockIdx.x * 256u + threadIdx.x) >> cpr_shift, H);
  }
  if (r.s >= Sq) return;
  const int64_t li = ((int64_t)r.b * H + r.h) * Sq + r.s;           // block lse: contiguous [B,H,Sq]
  const int64_t la_i = ((int64_t)r.b * H + r.h) * acc_lse_bh + r.s; // running lse: row pitch acc_lse_bh
  float* const ap = out_acc + r.b * as.b + r.h * as.h + (int64_t)r.s * as.s + ch * 4;
  float xb[8], xa[8];
  load44<T>(blk_out + r.b * bs.b + r.h * bs.h + (int64_t)r.s * bs.s + ch * 4, half, xb);
  const float lb = blk_lse[li];
  float la = 0.f;
  if (!INIT) {
    la = lse_acc[la_i];
    load44<float>(ap, half, xa);
  }
  float ln = lb;
  if (INIT) {
#pragma unroll
    for (int i = 0; i < 8; ++i) xa[i] = xb[i];
  } else {
    // w = sigmoid(lb - la); lse' = max + log1p(exp(-|lb - la|))
    const float d = lb - la;
    float w;
    if (d == d) {  // also covers +-inf on one side
      const float e = __expf(-fabsf(d));
      const float inv = 1.f / (1.f + e);
      w = d >= 0.f ? inv : e * inv;
      ln = fmaxf(la, lb) + log1pf(e);
    } else {  // both -inf: nothing accumulated on either side
      w = 0.f;
      ln = la;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) xa[i] = xa[i] - w * (xa[i] - xb[i]);
  }
  f32x4 a, b;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = xa[i];
    b[i] = xa[4 + i];
  }
  *(f32x4*)ap = a;
  *(f32x4*)(ap + half) = b;
  if (ch == 0) lse_acc[la_i] = ln;
}

template <typename T>
__global__ void __launch_bounds__(256) finalize_kernel(T* __restrict__ out, const float* __restrict__ out_acc,
                                                       int H, int cpr_shift, unsigned nrows, unsigned half,
                                                       Strides3 os, Strides3 as) {
  const unsigned gid = blockIdx.x * 256u + threadIdx.x;
  const unsigned row0 = gid >> cpr_shift;
  const int ch = (int)(gid & ((1u << cpr_shift) - 1u));
  float x[ROWS_PER_THREAD][8];
  T* op[ROWS_PER_THREAD];
  bool on[ROWS_PER_THREAD];
#pragma unroll
  for (int k = 0; k < ROWS_PER_THREAD; ++k) {
    const unsigned row = row0 + k * half;
    on[k] = row0 < half && row < nrows;
    const RowIdx r = decode_row(on[k] ? row : 0u, H);
    op[k] = out + r.b * os.b + r.h * os.h + (int64_t)r.s * os.s + ch * 8;
    if (on[k]) Load8<float>::ld(out_acc + r.b * as.b + r.h * as.h + (int64_t)r.s * as.s + ch * 8, x[k]);
  }
#pragma unroll
  for (int k = 0; k < ROWS_PER_THREAD; ++k)
    if (on[k]) Load8<T>::st(op[k], x[k]);
}

// Merge of the n block results a key-split forward left behind (rows j * Sq .. of `part`, [B, n * Sq, H, D] in P, and of
// part_lse, [B, H, n * Sq]): update_out_and_lse (sp_aurora/utils.py:103-104) over all of them at once, as a running
// (weighted sum, weight sum) relative to the largest lse so far.  A chunk whose scores are all -inf (lse -inf, no result) has no weight.
// Bound: the latency of its loads (a few rows, a few workgroups), so eight chunks are requested together.
template <typename T, typename P>
__global__ void __launch_bounds__(256) splitkv_combine_kernel(T* __restrict__ out, float* __restrict__ lse, const P* __restrict__ part,
                                                              const float* __restrict__ part_lse, int n, int H, int Sq, int D,
                                                              int cpr_shift, unsigned nrows, Strides3 os, int64_t lse_bh) {
  const unsigned gid = blockIdx.x * 256u + threadIdx.x;
  const unsigned row = gid >> cpr_shift;
  const int ch = (int)(gid & ((1u << cpr_shift) - 1u));
  if (row >= nrows) return;
  const RowIdx r = decode_row(row, H);
  const int64_t prow = (int64_t)H * D;                                  // elements between rows of `part`
  const P* pp = part + ((int64_t)r.b * n * Sq + r.s) * prow + r.h * D + ch * 8;
  const float* pl = part_lse + ((int64_t)r.b * H + r.h) * ((int64_t)n * Sq) + r.s;
  constexpr int NB = 8;
  float x[8], lb = -INFINITY, wsum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = 0.f;
  for (int j0 = 0; j0 < n; j0 += NB) {
    float xb[NB][8], l[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int j = j0 + u < n ? j0 + u : n - 1;
      l[u] = pl[(int64_t)j * Sq];
      Load8<P>::ld(pp + (int64_t)j * Sq * prow, xb[u]);
    }
    float mx = lb;
#pragma unroll
    for (int u = 0; u < NB; ++u) mx = fmaxf(mx, l[u]);
    const float ms = mx == -INFINITY ? 0.f : mx, wa = __expf(lb - ms);
    lb = mx;
    wsum *= wa;
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] *= wa;
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const bool none = j0 + u >= n || l[u] == -INFINITY;
      const float w = none ? 0.f : __expf(l[u] - ms);
      wsum += w;
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(none ? 0.f : xb[u][i], w, x[i]);
    }
  }
  const float inv = 1.f / wsum;
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] *= inv;
  Load8<T>::st(out + r.b * os.b + r.h * os.h + (int64_t)r.s * os.s + ch * 8, x);
  if (ch == 0) lse[((int64_t)r.b * H + r.h) * lse_bh + r.s] = lb + __logf(wsum);
}

// delta[b,h,s] = sum_d dout*out; the D/8 lanes of a row reduce with DPP-free shuffles.
template <typename T>
__global__ void __launch_bounds__(256) delta_kernel(const T* __restrict__ out, const T* __restrict__ dout,
                                                    float* __restrict__ delta, int H, int Sq, int cpr_shift,
                                                    unsigned nrows, unsigned half, Strides3 os, Strides3 ds) {
  const unsigned gid = blockIdx.x * 256u + threadIdx.x;
  const unsigned row0 = gid >> cpr_shift;
  const int cpr = 1 << cpr_shift;
  const int ch = (int)(gid & (unsigned)(cpr - 1));
  float a[ROWS_PER_THREAD][8], g[ROWS_PER_THREAD][8];
  int64_t di[ROWS_PER_THREAD];
  bool on[ROWS_PER_THREAD];
#pragma unroll
  for (int k = 0; k < ROWS_PER_THREAD; ++k) {
    const unsigned row = row0 + k * half;
    on[k] = row0 < half && row < nrows;
    const RowIdx r = decode_row(on[k] ? row : 0u, H);  // (rows past the end reread row 0: every lane takes part in the shuffles)
    di[k] = ((int64_t)r.b * H + r.h) * Sq + r.s;
    Load8<T>::ld(out + r.b * os.b + r.h * os.h + (int64_t)r.s * os.s + ch * 8, a[k]);
    Load8<T>::ld(dout + r.b * ds.b + r.h * ds.h + (int64_t)r.s * ds.s + ch * 8, g[k]);
  }
#pragma unroll
  for (int k = 0; k < ROWS_PER_THREAD; ++k) {
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc = __builtin_fmaf(a[k][i], g[k][i], acc);
    for (int off = cpr >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (on[k] && ch == 0) delta[di[k]] = acc;
  }
}

// Grid of the three kernels: x covers half the rows of one batch entry (a thread takes a row of
// each half), y the batch.
struct RowGrid {
  dim3 grid;
  unsigned nrows, half;
  int cpr_shift;
  bool ok;
};
RowGrid row_grid(int B, int H, int Sq, int D) {
  RowGrid g;
  const int64_t nrows = (int64_t)H * Sq;
  g.cpr_shift = __builtin_ctz((unsigned)(D / 8));
  g.ok = nrows < 0x7fffffffLL / (D / 8) && B <= 65535;
  g.nrows = (unsigned)nrows;
  g.half = (unsigned)((nrows + ROWS_PER_THREAD - 1) / ROWS_PER_THREAD);
  const int64_t threads = (int64_t)g.half * (D / 8);
  g.grid = dim3((unsigned)((threads + 255) / 256), (unsigned)B);
  return g;
}

}  // namespace

hipError_t spa_launch_merge(float* out_acc, float* lse_acc, const void* blk_out, const float* blk_lse, int B,
                            int H, int Sq, int D, Strides3 as, Strides3 bs, int dtype, int init,
                            int64_t acc_lse_bh, hipStream_t stream) {
  const RowGrid g = row_grid(B, H, Sq, D);
  if (!g.ok) return hipErrorInvalidValue;
  const int64_t blocks = ((int64_t)Sq * (D / 8) + 255) / 256 * H;
  const bool by_head = (int64_t)Sq * (D / 8) >= 256 && blocks * 256 <= 0x7fffffffLL;  // (fewer rows than a workgroup takes would leave threads idle)
  const dim3 grid = by_head ? dim3((unsigned)blocks, (unsigned)B) : g.grid;
#define SPA_MERGE(T, I)                                                                              \
  hipLaunchKernelGGL((merge_kernel<T, I>), grid, dim3(256), 0, stream, out_acc, lse_acc, (const T*)blk_out, \
                     blk_lse, H, Sq, g.cpr_shift, by_head, as, bs, acc_lse_bh)
  if (dtype == 0) { if (init) SPA_MERGE(float, true); else SPA_MERGE(float, false); }
  else if (dtype == 1) { if (init) SPA_MERGE(__bf16, true); else SPA_MERGE(__bf16, false); }
  else if (dtype == 2) { if (init) SPA_MERGE(_Float16, true); else SPA_MERGE(_Float16, false); }
  else return hipErrorInvalidValue;
#undef SPA_MERGE
  return hipGetLastError();
}

hipError_t spa_launch_finalize(void* out, const float* out_acc, int B, int H, int Sq, int D, Strides3 os,
                               Strides3 as, int dtype, hipStream_t stream) {
  const RowGrid g = row_grid(B, H, Sq, D);
  if (!g.ok) return hipErrorInvalidValue;
  if (dtype == 0)
    hipLaunchKernelGGL((finalize_kernel<float>), g.grid, dim3(256), 0, stream, (float*)out, out_acc, H, g.cpr_shift, g.nrows, g.half, os, as);
  else if (dtype == 1)
    hipLaunchKernelGGL((finalize_kernel<__bf16>), g.grid, dim3(256), 0, stream, (__bf16*)out, out_acc, H, g.cpr_shift, g.nrows, g.half, os, as);
  else if (dtype == 2)
    hipLaunchKernelGGL((finalize_kernel<_Float16>), g.grid, dim3(256), 0, stream, (_Float16*)out, out_acc, H, g.cpr_shift, g.nrows, g.half, os, as);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t spa_launch_delta(const void* out, const void* dout, float* delta, int B, int H, int Sq, int D,
                            Strides3 os, Strides3 ds, int dtype, hipStream_t stream) {
  const RowGrid g = row_grid(B, H, Sq, D);
  if (!g.ok) return hipErrorInvalidValue;
  if (dtype == 0)
    hipLaunchKernelGGL((delta_kernel<float>), g.grid, dim3(256), 0, stream, (const float*)out, (const float*)dout, delta, H, Sq, g.cpr_shift, g.nrows, g.half, os, ds);
  else if (dtype == 1)
    hipLaunchKernelGGL((delta_kernel<__bf16>), g.grid, dim3(256), 0, stream, (const __bf16*)out, (const __bf16*)dout, delta, H, Sq, g.cpr_shift, g.nrows, g.half, os, ds);
  else if (dtype == 2)
    hipLaunchKernelGGL((delta_kernel<_Float16>), g.grid, dim3(256), 0, stream, (const _Float16*)out, (const _Float16*)dout, delta, H, Sq, g.cpr_shift, g.nrows, g.half, os, ds);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// part32: `part` is fp32, not of the element type.
hipError_t spa_launch_splitkv_combine(void* out, float* lse, const void* part, const float* part_lse, int n, int B, int H, int Sq,
                                      int D, Strides3 os, int64_t lse_bh, int dtype, bool part32, hipStream_t stream) {
  const RowGrid g = row_grid(B, H, Sq, D);
  if (!g.ok || n < 1 || (dtype != 1 && dtype != 2)) return hipErrorInvalidValue;
#define SPA_COMBINE(T, P)                                                                                                                              \
  hipLaunchKernelGGL((splitkv_combine_kernel<T, P>), g.grid, dim3(256), 0, stream, (T*)out, lse, (const P*)part, part_lse, n, H, Sq, D, g.cpr_shift, \
                     g.nrows, os, lse_bh)
  if (dtype == 1) {
    if (part32) SPA_COMBINE(__bf16, float); else SPA_COMBINE(__bf16, __bf16);
  } else {
    if (part32) SPA_COMBINE(_Float16, float); else SPA_COMBINE(_Float16, _Float16);
  }
#undef SPA_COMBINE
  return hipGetLastError();
}
