// Block-wise attention backward for gfx950 with the GLOBAL lse / delta of the query rows:
//   P = exp(q k^T * scale + mask - lse);  dV += P^T dO;  dP = dO V^T;
//   dS = P * (dP - delta);  dQ += dS K * scale;  dK += dS^T Q * scale.
// Stands in for the per-step body of intel_ring_flash_attn_backward
// (sp_aurora/intel_ring_flash_attn.py:192-258), which re-runs autograd on each block.
//
// Two kernels, no atomics, every output row has one owner (deterministic):
//   dq kernel   : workgroup = 64, 128 or 256 query rows, walks key tiles of 64: 4 or 8 waves of 32 rows, or half as many rows and
//                 pairs of waves that share 32 rows and each take half of a tile's keys (dq_form, KG).
//                 S^T = K Q^T and dP^T = V dO^T land with a lane owning one query row,
//                 so lse/delta are per-lane scalars and dS^T is, register for register,
//                 the B operand of dQ^T = K^T dS^T.
//   dkdv kernel : workgroup = 128 keys (4 waves x 32), walks query tiles of 64; or 64 keys, pairs of waves sharing 32 (keys_64, QG).
//                 S = Q K^T and dP = dO V^T land with a lane owning one key, so P and dS
//                 are the B operands of dV^T = dO^T P and dK^T = Q^T dS.
//
// Streamed tiles (K, V / Q, dO; 64 rows) travel from global memory straight into LDS, several
// tiles ahead, rows back to back with their 16-byte chunks XOR-permuted so that both ways of
// reading a tile run without bank conflicts: rows as 16-byte reads (A operands of the S / dP
// contractions) and, through the transposing read, columns (A operands K^T, Q^T, dO^T of the
// gradient contractions).  No transposed copies exist.
//
// D = 128: one wave per SIMD (the 8-wave dq kernel: two, which also halves the K/V traffic per query row).  D <= 64: both
// kernels fit two 4-wave workgroups to a CU (256 registers a lane); one covers the other's start, end and LDS latency:
// [2,4096,32,64] causal backward 582 -> 480 us, [64,512,16,64] 312 -> 243 us.
// Software-pipelined inside the wave at half-tile (32 rows) granularity:
// the MFMAs that produce S and dP of half-tile g+1 are interleaved, one to one, with the
// element-wise work (exp, dS) on half-tile g, followed by the gradient MFMAs of half-tile g; in the dk/dv kernel the
// gradient MFMAs stand between the others as well, so that vector work and matrix work are spread alike over the whole pass.
// MFMA operands come from LDS through a rolling window that runs ahead of the MFMAs and is
// carried across loop iterations; one workgroup barrier per 64-row tile.
// Accumulators are fp32 in HBM and are ADDED to (read-modify-write by the owning lane).
// In the one-wave-per-SIMD kernels the MFMAs are written with their register files spelled out
// (gradient accumulators in AGPRs, S / dP tiles in VGPRs), see MmaAsm.
#include "spa_common.h"
#include "spa_host.h"
#include <math.h>
#include <stdlib.h>

namespace {

constexpr int BWD_THREADS = 256;
constexpr int BWD_ROWS = 64;    // rows (keys or queries) per streamed LDS tile
constexpr int BWD_STAGES = 4;   // tiles resident or on their way
constexpr int BWD_LOOK_MAX = 8; // operands are fetched from LDS up to this many MFMAs ahead
constexpr unsigned OFF_NONE = 0x80000000u;  // a buffer offset beyond any tensor: the load stores zeros

template <int D, int THREADS = BWD_THREADS>
struct BwdCfg {
  static constexpr int ROWB = D * 2;             // bytes per tile row
  static constexpr int TILEB = BWD_ROWS * ROWB;  // one tile
  static constexpr int CPR = D / 8;              // 16-byte chunks per row
  static constexpr int NDMA = TILEB / (THREADS * 16);  // direct loads per thread and tile
  static_assert(NDMA >= 1, "a tile must give every thread at least one 16-byte slot");
  static constexpr int RPD = THREADS / CPR;  // rows one round of the workgroup's loads covers
};

// Chunk permutation of a tile row, good for both read patterns: 16 consecutive rows at one chunk
// index fall into 16 different 16-byte bank groups, and so do the 4 rows x 4 chunks a half wave
// covers with one transposing read.  Depends on row % 16 only.
template <int D>
__device__ __forceinline__ int tile_swizzle(int row) {
  return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3)
         : D == 64 ? (((row >> 1) & 1) << 2) | ((row >> 2) & 3)
                   : (row >> 2) & 3;
}

// Per-lane LDS offsets (relative to a tile) of the two read patterns.
template <int D>
struct TileReads {
  unsigned row[D / 16];     // chunk 2 ks + hh of row ln (+ 32 rows: second half)
  unsigned tr[D / 32][2];   // transposing read of 4 dims of row 8 h8 + 4 hh + e (+ 16 u rows, + 32 rows)
  __device__ __forceinline__ void init(int lane) {
    typedef BwdCfg<D> C;
    const int ln = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) row[ks] = ln * C::ROWB + (((2 * ks + hh) ^ tile_swizzle<D>(ln)) * 16);
    const int blk = lane >> 4, e = (lane >> 2) & 3, c4 = lane & 3;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int h8 = 0; h8 < 2; ++h8) {
        const int r = 8 * h8 + 4 * hh + e;
        const int chunk = db * 4 + (blk & 1) * 2 + (c4 >> 1);
        tr[db][h8] = r * C::ROWB + ((chunk ^ tile_swizzle<D>(r)) * 16) + (c4 & 1) * 8;
      }
  }
};

// Global side of the direct loads: thread tid owns 16-byte slot tid of every round of 256 slots;
// round j covers rows j * RPD + tid / CPR.  Slot (row, pos) receives chunk pos ^ swizzle(row).
// ADDR_BIG: the tensor's rows of one (batch, head) may span 2 GiB or more; the descriptor is re-based per tile
// (buffer_window) instead of covering the whole tensor.  ADDR_MAP: the rows lie in shards (RowMap): every lane looks up
// its row (about 15 vector instructions per load), or, for the tiles that are streamed, ShardTiles finds the rows of a whole tile.
enum { ADDR_PLAIN = 0, ADDR_BIG = 1, ADDR_MAP = 2 };
template <typename T, int D, int THREADS = BWD_THREADS, int ADDR = ADDR_PLAIN>
struct TileLoader {
  u32x4 rsrc;
  unsigned lane_off;  // bytes
  unsigned row_b;     // bytes per tensor row
  const T* base_;             // ADDR_BIG only
  unsigned long long total_;  // ADDR_BIG only: bytes from base_ to the end of the last row
  int rows_, drow_;           // ADDR_MAP only
  unsigned row_off_;          // ADDR_MAP only: bytes from the tile's (or round's) first row to this thread's
  // rows: rows of the sequence; span: rows of the tensor from base to the sequence's last row
  __device__ __forceinline__ void init(const T* base, int64_t row_stride, int rows, int span, int tid) {
    typedef BwdCfg<D, THREADS> C;
    total_ = (unsigned long long)((((int64_t)span - 1) * row_stride + D) * (int64_t)sizeof(T));
    base_ = base;
    rsrc = buffer_descriptor(base, ADDR == ADDR_BIG ? 0u : (unsigned)total_);  // (ADDR_BIG: an empty range, for tiles that are not wanted)
    const int drow = tid / C::CPR, dpos = tid % C::CPR;
    rows_ = rows;
    drow_ = drow;
    row_off_ = (unsigned)(drow * row_stride * (int64_t)sizeof(T));
    lane_off = (unsigned)(((ADDR == ADDR_MAP ? 0 : drow * row_stride) + ((dpos ^ tile_swizzle<D>(drow)) * 8)) * (int64_t)sizeof(T));
    row_b = (unsigned)(row_stride * (int64_t)sizeof(T));
  }
  // round q of the tile whose first row is row0 (on = false: store zeros) into LDS at lds_wave
  __device__ __forceinline__ void load(int q, bool on, int row0, unsigned lds_wave, const RowMap& map, int pitch) const {
    typedef BwdCfg<D, THREADS> C;
    if constexpr (ADDR == ADDR_MAP) {
      const int r = row0 + q * C::RPD + drow_;
      const unsigned off = lane_off + (unsigned)map.at(r, pitch) * row_b;
      load_to_lds_b128(rsrc, on && r < rows_ ? off : OFF_NONE, lds_wave + q * (THREADS * 16));
    } else if constexpr (ADDR == ADDR_BIG) {
      unsigned rel = OFF_NONE;
      u32x4 rs = rsrc;
      if (on) rs = buffer_window(base_, total_, (unsigned long long)(unsigned)row0 * row_b, rel);
      load_to_lds_b128(rs, lane_off + rel + (unsigned)(q * C::RPD) * row_b, lds_wave + q * (THREADS * 16));
    } else {
      const unsigned u = on ? (unsigned)(row0 + q * C::RPD) * row_b : OFF_NONE;
      load_to_lds_b128(rsrc, lane_off + u, lds_wave + q * (THREADS * 16));
    }
  }
};

// The tiles of 64 rows of a pair of tensors with rows in shards, one after the other.  Where a segment has 64 rows or more a tile touches
// two of them at most: which two is the same for all lanes, and a lane's row is in the first or the second.  (Looked up row by row the
// one-wave dk/dv kernel, which issues an instruction every four clocks, spent 135 of 650 per tile on it.)
template <typename T, int D, int THREADS>
struct ShardTiles {
  typedef BwdCfg<D, THREADS> C;
  typedef TileLoader<T, D, THREADS, ADDR_MAP> Loader;
  int seg, seg_end;                      // segment of the tile's first row, and where it ends
  unsigned at[2][C::NDMA], stat_at;      // byte offsets of this thread's loads, and of the lane's row in lse and delta
  __device__ __forceinline__ void init(const RowMap& map, int row0) {
    seg = __builtin_amdgcn_readfirstlane(map.segment(row0));
    seg_end = (seg + 1) * map.L;
  }
  // (called once for every tile, in order)
  __device__ __forceinline__ void find(const RowMap& map, const ShardMap& m, int row0, int rows, const Loader& a, const Loader& b, int lane, bool on) {
    if (map.L >= BWD_ROWS) {
      if (row0 >= seg_end) {
        ++seg;
        seg_end += map.L;
      }
      const bool two = on && seg_end < rows;
      const int r1 = row0 + map.shift(seg, m.pitch), r2 = row0 + map.shift(seg + 1, m.pitch);
#pragma unroll
      for (int q = 0; q < C::NDMA; ++q) {
        const bool first = row0 + q * C::RPD + a.drow_ < seg_end;
        const unsigned a1 = on ? (unsigned)(r1 + q * C::RPD) * a.row_b : OFF_NONE, a2 = two ? (unsigned)(r2 + q * C::RPD) * a.row_b : OFF_NONE;
        const unsigned b1 = on ? (unsigned)(r1 + q * C::RPD) * b.row_b : OFF_NONE, b2 = two ? (unsigned)(r2 + q * C::RPD) * b.row_b : OFF_NONE;
        at[0][q] = a.lane_off + a.row_off_ + (first ? a1 : a2);
        at[1][q] = b.lane_off + b.row_off_ + (first ? b1 : b2);
      }
      const unsigned s1 = on ? (unsigned)(row0 + map.shift(seg, m.lse_pitch)) * 4u : OFF_NONE;
      const unsigned s2 = two ? (unsigned)(row0 + map.shift(seg + 1, m.lse_pitch)) * 4u : OFF_NONE;
      stat_at = lane * 4 + (row0 + lane < seg_end ? s1 : s2);
    } else {
#pragma unroll
      for (int q = 0; q < C::NDMA; ++q) {
        const int r = row0 + q * C::RPD + a.drow_, to = map.at(r, m.pitch);
        at[0][q] = on && r < rows ? a.lane_off + (unsigned)to * a.row_b : OFF_NONE;
        at[1][q] = on && r < rows ? b.lane_off + (unsigned)to * b.row_b : OFF_NONE;
      }
      stat_at = on && row0 + lane < rows ? (unsigned)map.at(row0 + lane, m.lse_pitch) * 4u : OFF_NONE;
    }
  }
  // behind the last tile: the first tensor's rows once more, zeros for the others
  __device__ __forceinline__ void repeat_first() {
#pragma unroll
    for (int q = 0; q < C::NDMA; ++q) at[1][q] = OFF_NONE;
    stat_at = OFF_NONE;
  }
};

// The lane's operands of ROWS = 32 resident rows (row ln; 16 bytes per 16-deep contraction step) out of rows that were
// loaded like a tile.  Straight from memory they are 16-byte pieces of 32 rows per load instruction: 32 cache lines for 1 KB,
// and the first 5 us of a workgroup went into them; as a tile every instruction reads whole rows.
template <typename F, int D>
__device__ __forceinline__ void read_rows(F (&f)[D / 16], unsigned rows_at, const TileReads<D>& rd) {
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) f[ks] = as_frag<F>(lds_read_b128(rows_at + rd.row[ks]));
}

// Writes the wave's 32 rows of a gradient (accumulator layout: a lane holds, of row ln, dims 32 db + 8 g + 4 hh .. + 3) in T.
// Through LDS (32 rows of the wave's own, chunks XOR-permuted), so that a store instruction writes whole rows: the 8-byte
// pieces a lane holds are 32 cache lines per instruction, and the last 6 us of a workgroup went into them.
// n_rows: rows that exist from the wave's first row on; row(r): where row r of the wave's goes.
template <typename T, int D, typename Row>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[D / 32], float scale, Row&& row, int n_rows, unsigned char* lds, int lane) {
  constexpr int CPR = D / 8;  // 16-byte chunks per row
  const int ln = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      u32x2 st;
      st[0] = Mma16<T>::pack2(acc[db][4 * g + 0] * scale, acc[db][4 * g + 1] * scale);
      st[1] = Mma16<T>::pack2(acc[db][4 * g + 2] * scale, acc[db][4 * g + 3] * scale);
      *(u32x2*)(lds + ln * (D * 2) + (((db * 4 + g) ^ (ln & (CPR - 1))) * 16) + 8 * hh) = st;
    }
  // (the wave's own LDS writes are visible to its later reads)
#pragma unroll
  for (int i = 0; i < 32 * CPR / 64; ++i) {
    const int r = i * (64 / CPR) + lane / CPR, ch = lane % CPR;
    const u32x4 x = *(const u32x4*)(lds + r * (D * 2) + ((ch ^ (r & (CPR - 1))) * 16));
    if (r < n_rows) *(u32x4*)((T*)row(r) + ch * 8) = x;
  }
}

// One MFMA operand from two transposing reads (rows 0..3 and 8..11 of a lane's group of 16).
template <typename F>
__device__ __forceinline__ F frag_tr(unsigned addr_lo, unsigned addr_hi) {
  const u32x2 r0 = lds_read_tr16_b64(addr_lo);
  const u32x2 r1 = lds_read_tr16_b64(addr_hi);
  u32x4 x;
  x[0] = r0[0];
  x[1] = r0[1];
  x[2] = r1[0];
  x[3] = r1[1];
  return as_frag<F>(x);
}

__device__ __forceinline__ void zero16(f32x16& x) {
#pragma unroll
  for (int v = 0; v < 16; ++v) x[v] = 0.f;
}

template <int N>
__device__ __forceinline__ void wait_loads_but() {  // until at most N of this wave's loads are in flight
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// The barrier without the waits of __syncthreads(), which would drain the operands in flight: the caller has waited for what it needs.  The compiler
// knows no memory access of s_barrier; the empty assembly keeps loads and stores on their side of it, and a sched_barrier(0) follows in the loops.
__device__ __forceinline__ void barrier_alone() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// MFMAs with the accumulator's register file spelled out.  The compiler gives every MFMA of a
// function the same form; the one-wave-per-SIMD kernels want both: the gradient accumulators
// (touched by MFMAs only) in AGPRs, the S / dP tiles, which the VALU works on, in VGPRs, so that
// no v_accvgpr_read / v_accvgpr_write copies are needed between the matrix pipe and the VALU.
// The compiler does not see these as MFMAs: the code keeps the distances the hardware needs (srcC is the
// destination itself or the literal 0, never a register a VALU instruction has just written).  A VALU read of a tile needs 11 wait states after
// the tile's last MFMA, which takes the matrix pipe for 8 passes: with MFMA_APART others issued in between, each of which had to wait for the one
// before it, at least 16 have gone by.  The loops' orders are held to that by static_asserts: 8 gradient MFMAs in the dq kernel, 3 MFMAs in the
// dk/dv kernel.  Where no others follow, mfma_settle() waits.
constexpr int MFMA_APART = 2;
template <typename T>
struct MmaAsm;
template <>
struct MmaAsm<__bf16> {
  typedef bf16x8 frag;
  static __device__ __forceinline__ void first_v(f32x16& c, frag a, frag b) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void acc_v(f32x16& c, frag a, frag b) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void acc_a(f32x16& c, frag a, frag b) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
};
template <>
struct MmaAsm<_Float16> {
  typedef f16x8 frag;
  static __device__ __forceinline__ void first_v(f32x16& c, frag a, frag b) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void acc_v(f32x16& c, frag a, frag b) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void acc_a(f32x16& c, frag a, frag b) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
};

// ------------------------------------------------------------------------------------------
// dQ kernel
// ------------------------------------------------------------------------------------------
// KG = 2: the waves come in two groups that own the same query rows, and each takes 32 of a tile's 64 keys; their sums are added through LDS.
template <int D, int NW = 4, int KG = 1>
struct DqCfg {
  typedef BwdCfg<D, NW * 64> C;
  static constexpr int ROWS = NW / KG * 32;   // query rows of a workgroup
  static constexpr int STAGES = KG == 2 ? 5 : BWD_STAGES;
  static constexpr int STAGE = 2 * C::TILEB;  // K tile, V tile
  static constexpr int SMEM = STAGES * STAGE;
  static constexpr int NL = 2 * C::NDMA;      // loads per thread and stage
};

// Variable-length batch: sequence b owns rows cu_q[b] .. cu_q[b+1] of the query-side tensors and
// cu_k[b] .. cu_k[b+1] of the key-side ones; the kernel then works on that sequence as on batch 0
// of a batch whose bases and sizes are the sequence's.
// map: set up for the sequence's rows where they lie in shards (the sequence is then p.map.P times as long as cu says).
template <typename T>
__device__ __forceinline__ void select_sequence(BwdParams& p, int& b, RowMap& map) {
  if (!p.cu_q) {
    if (p.map.P) map.init(p.map, p.Sq / p.map.P);
    return;
  }
  const int q_lo = p.cu_q[b], k_lo = p.cu_k[b];
  p.Sq = p.cu_q[b + 1] - q_lo;
  p.Sk = p.cu_k[b + 1] - k_lo;
  p.q = (const T*)p.q + (int64_t)q_lo * p.qs.s;
  p.dout = (const T*)p.dout + (int64_t)q_lo * p.dos.s;
  p.k = (const T*)p.k + (int64_t)k_lo * p.ks.s;
  p.v = (const T*)p.v + (int64_t)k_lo * p.vs.s;
  const int64_t gsz = p.grads_in_t ? (int64_t)sizeof(T) : 4;  // gradients written in T, or fp32 accumulators
  p.dq = (float*)((char*)p.dq + q_lo * p.dqs.s * gsz);
  p.dk = (float*)((char*)p.dk + k_lo * p.dks.s * gsz);
  p.dv = (float*)((char*)p.dv + k_lo * p.dvs.s * gsz);
  if (p.out) p.out = (const T*)p.out + (int64_t)q_lo * p.os.s;
  p.lse += q_lo;
  p.delta += q_lo;
  b = 0;
  if (p.map.P) {
    map.init(p.map, p.Sq);
    p.Sq *= p.map.P;
    p.Sk = p.Sq;
  }
}

// The (batch or sequence, head) and the tile (of `rows` query rows, or keys) of a workgroup: pairs first, in groups
// (spa_head_groups), or, for a packed batch with a numbered grid, heads first and then the tiles of all sequences (sequence_tile).  The
// tiles that see the most of the other side go first: with a causal mask the last query tiles and the first key tiles.
__device__ __forceinline__ bool workgroup_tile(const BwdParams& p, bool queries, int rows, int lane, int& b, int& h, int& tile) {
  int n;
  if (p.numbered) {
    const int number = blockIdx.x / p.H;
    h = blockIdx.x - number * p.H;
    if (!sequence_tile(queries ? p.cu_q : p.cu_k, p.B, p.map.P ? p.map.P : 1, rows, number, lane, b, tile, n)) return false;
  } else {
    const int pair = blockIdx.x + blockIdx.z * gridDim.x;
    if (pair >= p.B * p.H) return false;
    h = pair % p.H;
    b = pair / p.H;
    tile = blockIdx.y;
    n = gridDim.y;
  }
  if (queries) tile = n - 1 - tile;
  return true;
}

// A row of a gradient that is written (BwdParams::grads_in_t) and that no tile contributes to: the
// lane's share of the row (the columns the epilogues give it) is set to zero.
template <typename E, int D>
__device__ __forceinline__ void zero_grad_row(E* rowp, int hh) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if constexpr (sizeof(E) == 2) {
        const u32x2 z = {0u, 0u};
        *(u32x2*)(rowp + db * 32 + 8 * g + 4 * hh) = z;
      } else {
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        *(f32x4*)(rowp + db * 32 + 8 * g + 4 * hh) = z;
      }
    }
}

template <typename T, int D, int NW, int ADDR = ADDR_PLAIN, int KG = 1>
__global__ void __launch_bounds__(NW * 64, NW == 4 && D <= 64 ? 2 : 1) flash_bwd_dq_kernel(const BwdParams pk) {
  BwdParams p = pk;  // a variable-length batch rewrites the sizes and bases for its sequence below
  typedef BwdCfg<D, NW * 64> C;
  typedef DqCfg<D, NW, KG> G;
  typedef Mma16<T> M;
  typedef MmaAsm<T> MA;
  // one wave per SIMD: AGPRs are there for the dq accumulators (D = 128; two workgroups to a CU at smaller D)
  constexpr bool MIXED = NW == 4 && D == 128;
  typedef typename M::frag frag;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  int b, h, qt;
  if (!workgroup_tile(p, true, G::ROWS, lane, b, h, qt)) return;
  const int q0 = qt * G::ROWS;
  constexpr int RG = NW / KG;            // groups of 32 rows
  const int rg = w % RG, kg = w / RG;    // the wave's rows, and its half of the keys of a tile
  const int qw0 = q0 + rg * 32;
  RowMap map = {};
  select_sequence<T>(p, b, map);
  constexpr bool MAP = ADDR == ADDR_MAP;
  auto row_of = [&](int r) { return MAP ? map.at(r, p.map.pitch) : r; };        // where row r of the sequence lies
  auto stat_of = [&](int r) { return MAP ? map.at(r, p.map.lse_pitch) : r; };   // in lse and delta
  // rows of the tensors from the sequence's first to its last
  const int span_q = MAP ? (p.map.P - 1) * p.map.pitch + p.Sq / p.map.P : p.Sq, span_k = MAP ? span_q : p.Sk;
  if (q0 >= p.Sq || p.Sk <= 0) {  // (variable-length batches only) no keys: nothing to add to dq, a written dq is zero
    if (p.grads_in_t && qw0 + ln < p.Sq)
      zero_grad_row<T, D>((T*)p.dq + b * p.dqs.b + h * p.dqs.h + (int64_t)row_of(qw0 + ln) * p.dqs.s, hh);
    return;
  }

  const T* qp = (const T*)p.q + b * p.qs.b + h * p.qs.h;
  const T* kp = (const T*)p.k + b * p.ks.b + h * p.ks.h;
  const T* vp = (const T*)p.v + b * p.vs.b + h * p.vs.h;
  const T* dop = (const T*)p.dout + b * p.dos.b + h * p.dos.h;

  const int qrow = qw0 + ln;
  const int qrow_c = qrow < p.Sq ? qrow : p.Sq - 1;

  frag qf[D / 16], dof[D / 16];
  const int64_t li = ((int64_t)b * p.H + h) * p.lse_bh + stat_of(qrow_c);
  const float l2 = p.lse[li] * 1.4426950408889634f;
  const float c = p.scale_log2;
  const float hidden = c < 0.f ? INFINITY : -INFINITY;  // a hidden score: exp2(hidden * c - lse) = 0 for either sign of the scale
  const int lim = p.causal ? (qrow < p.Sk - 1 ? qrow : p.Sk - 1) : p.Sk - 1;  // last visible key

  const int kv_end = p.causal ? (q0 + G::ROWS < p.Sk ? q0 + G::ROWS : p.Sk) : p.Sk;
  const int nt = (kv_end + BWD_ROWS - 1) / BWD_ROWS;  // key tiles this workgroup visits

  TileLoader<T, D, NW * 64, ADDR> kld, vld;
  kld.init(kp, p.ks.s, p.Sk, span_k, tid);
  vld.init(vp, p.vs.s, p.Sk, span_k, tid);
  TileReads<D> rd;
  rd.init(lane);
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_u8*)smem;
  auto stage_of = [&](int i) { return lds0 + (unsigned)i % G::STAGES * G::STAGE; };
  ShardTiles<T, D, NW * 64> tiles;
  if constexpr (MAP) tiles.init(map, 0);
  auto issue_one = [&](int i, int n) {  // load n of tile i's G::NL (in order): K, then V -> its stage
    const unsigned dst = stage_of(i) + w * 1024;
    if constexpr (MAP) {
      if (n == 0) tiles.find(map, p.map, i * BWD_ROWS, p.Sk, kld, vld, lane, i < nt);
      const int t = n / C::NDMA, q = n % C::NDMA;
      load_to_lds_b128(t ? vld.rsrc : kld.rsrc, tiles.at[t][q], dst + t * C::TILEB + q * (NW * 64 * 16));
    } else if (n < C::NDMA) {
      kld.load(n, i < nt, i * BWD_ROWS, dst, map, p.map.pitch);
    } else {
      vld.load(n - C::NDMA, i < nt, i * BWD_ROWS, dst + C::TILEB, map, p.map.pitch);
    }
  };
  auto issue_tile = [&](int i) {
#pragma unroll
    for (int n = 0; n < G::NL; ++n) issue_one(i, n);
  };

  f32x16 dq[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) zero16(dq[i]);

  // Half-tile g = 2 i + t is keys [32 g, 32 g + 32).  One pass of the loop body handles tile i:
  //   list 2i  : S^T, dP^T of half 2i+1 (tile i, rows 32..63)   | dS^T of half 2i   | dQ of half 2i
  //   list 2i+1: S^T, dP^T of half 2i+2 (tile i+1, rows 0..31)  | dS^T of half 2i+1 | dQ of half 2i+1
  // NA MFMAs produce, the element-wise work rides between them, NB MFMAs consume.  KG = 2: one list a pass, on the wave's half of tile i, with
  // S^T, dP^T of its half of tile i + 1 (and the first operands of that of tile i + 2, hence a stage more).
  constexpr int LISTS = 2 / KG;
  constexpr int NA = 2 * (D / 16), NB = 2 * (D / 32), NLIST = NA + NB, NBODY = LISTS * NLIST;
  constexpr int LOOK_CAP = NW == 8 || D <= 64 ? 4 : BWD_LOOK_MAX;  // two waves per SIMD: 256 registers each, and the other wave covers LDS latency
  constexpr int BWD_LOOK = NA < LOOK_CAP ? NA : LOOK_CAP;
  static_assert(NBODY % BWD_LOOK == 0 && BWD_LOOK <= NA, "the operand window must tile the loop body");
  static_assert(!MIXED || NB >= MFMA_APART, "the gradient MFMAs stand between a tile's last MFMA and its element-wise work");

  // The workgroup's rows of q and dout pass through the stages on their way into registers, and those of out, which give
  // delta = rowsum(dout * out) (written for the dk / dv kernel).  128 rows are one stage a tensor: all of them and the first tile are
  // requested together (KG = 2: the first two tiles).  256 rows are two: out follows when q and dout have been read, with the first two tiles.
  constexpr bool TOGETHER = RG <= 4;
  constexpr int FIRST = KG;   // (TOGETHER) tiles requested with the rows
  constexpr int RT = RG / 2;  // tiles of 64 rows
  const unsigned own = (rg >> 1) * C::TILEB + (rg & 1) * 32 * C::ROWB;
  const unsigned q_at = lds0 + (TOGETHER ? 2 * G::STAGE : 0), do_at = lds0 + (TOGETHER ? 3 : 2) * G::STAGE;
  const unsigned out_at = lds0 + (KG == 2 ? 4 : TOGETHER ? 1 : 2) * G::STAGE;
  auto load_rows = [&](const T* base, int64_t stride, unsigned dst) {
    TileLoader<T, D, NW * 64, ADDR> ld;
    ld.init(base, stride, p.Sq, span_q, tid);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int q = 0; q < C::NDMA; ++q) ld.load(q, q0 + i * BWD_ROWS < p.Sq, q0 + i * BWD_ROWS, dst + i * C::TILEB + w * 1024, map, p.map.pitch);
  };
  auto load_out = [&]() {
    if (p.out) load_rows((const T*)p.out + b * p.os.b + h * p.os.h, p.os.s, out_at);
  };
  load_rows(qp, p.qs.s, q_at);
  load_rows(dop, p.dos.s, do_at);
  if constexpr (TOGETHER) {
    load_out();
#pragma unroll
    for (int i = 0; i < FIRST; ++i) issue_tile(i);
    wait_loads_but<FIRST * G::NL>();
  } else {
    wait_loads_but<0>();
  }
  __syncthreads();
  read_rows<frag, D>(qf, q_at + own, rd);
  read_rows<frag, D>(dof, do_at + own, rd);
  if constexpr (!TOGETHER) {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): read ...
    __syncthreads();                     // ... by every wave
    load_out();
    issue_tile(0);
    issue_tile(1);
  }
  float dl;
  if (p.out) {
    if constexpr (!TOGETHER) {
      wait_loads_but<2 * G::NL>();
      __syncthreads();
    }
    float sum = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const u32x4 x = lds_read_b128(out_at + own + rd.row[ks]), y = __builtin_bit_cast(u32x4, dof[ks]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x0, x1, y0, y1;
        M::unpack2(x[i], x0, x1);
        M::unpack2(y[i], y0, y1);
        sum = __builtin_fmaf(x1, y1, __builtin_fmaf(x0, y0, sum));
      }
    }
    dl = halves_sum(sum);
    if (hh == 0 && qrow < p.Sq && kg == 0) p.delta[li] = dl;
  } else {
    dl = p.delta[li];
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);  // the rows have been read ...
  __syncthreads();                     // ... by every wave
  if constexpr (TOGETHER) issue_tile(FIRST);
  issue_tile(FIRST + 1 > 2 ? FIRST + 1 : 2);
  wait_loads_but<2 * G::NL>();
  __syncthreads();
  constexpr int AHEAD = KG == 2 ? 4 : 3;  // tile i + AHEAD is requested in pass i
  const unsigned half = KG == 2 ? kg * 32 * C::ROWB : 0;  // the wave's half of a tile

  f32x16 sc, dc, sn, dn;  // S^T, dP^T of the current / next half-tile
  {
    if (!MIXED) {
      zero16(sc);
      zero16(dc);
    }
    const unsigned kb = stage_of(0) + half;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const frag a0 = as_frag<frag>(lds_read_b128(kb + rd.row[ks]));
      const frag a1 = as_frag<frag>(lds_read_b128(kb + C::TILEB + rd.row[ks]));
      if (MIXED) {
        if (ks == 0) {
          MA::first_v(sc, a0, qf[0]);
          MA::first_v(dc, a1, dof[0]);
        } else {
          MA::acc_v(sc, a0, qf[ks]);
          MA::acc_v(dc, a1, dof[ks]);
        }
      } else {
        sc = M::run(a0, qf[ks], sc);
        dc = M::run(a1, dof[ks], dc);
      }
    }
  }

  // operand fetch number J of the body of tile i (J >= NBODY: the first operands of the next body)
  unsigned row_cur[D / 16], row_nxt[D / 16], tr_cur[D / 32][2];
  // KG = 2: row_cur and tr_cur are moved on to the next tile where that is first read through them; stages of tiles i - 1 .. i + 2
  unsigned st_before = stage_of(0), st_this = st_before, st_next = stage_of(1), st_after = stage_of(2);
  auto advance = [&](unsigned& at, unsigned by) {
    at += by;
    asm volatile("" : "+v"(at));  // (kept, not formed again from the tile's number at every use)
  };
  auto set_addresses = [&](int i) {
    const unsigned a = stage_of(i), n = stage_of(i + 1);
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      row_cur[ks] = a + rd.row[ks];
      row_nxt[ks] = n + rd.row[ks];
    }
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int h8 = 0; h8 < 2; ++h8) tr_cur[db][h8] = a + rd.tr[db][h8];
  };
  auto fetch = [&](int J) -> frag {
    const int body = J / NBODY, j2 = J % NBODY;
    const int list = j2 / NLIST, j = j2 % NLIST;
    if (j < NA) {  // j = 2 ks + which: K row (S^T) or V row (dP^T) of the half-tile being produced
      const int ks = j >> 1, which = j & 1;
      if constexpr (KG == 2) {
        // the wave's rows of tile i+1; of the next body, tile i+2
        if (which == 0) advance(row_cur[ks], body ? st_after - st_next : st_next - st_this);
        return as_frag<frag>(lds_read_b128(row_cur[ks] + which * C::TILEB));
      }
      // list 0 of this body: tile i rows 32..; list 1: tile i+1 rows 0..; list 0 of the next body: tile i+1 rows 32..
      const unsigned base = (body == 0 && list == 0) ? row_cur[ks] + 32 * C::ROWB
                            : (body == 0)           ? row_nxt[ks]
                                                    : row_nxt[ks] + 32 * C::ROWB;
      return as_frag<frag>(lds_read_b128(base + which * C::TILEB));
    }
    const int jb = j - NA;  // jb = u * (D/32) + db : K^T operand of half-tile `list` of tile i
    const int db = jb % (D / 32), u = jb / (D / 32);
    if (KG == 2 && u == 0) {
#pragma unroll
      for (int h8 = 0; h8 < 2; ++h8) advance(tr_cur[db][h8], st_this - st_before);
    }
    const unsigned off = (list * 32 + u * 16) * C::ROWB;
    return frag_tr<frag>(tr_cur[db][0] + off, tr_cur[db][1] + off);
  };

  frag win[BWD_LOOK];
  frag dsf[2];
  set_addresses(0);
  if constexpr (KG == 2) {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) row_cur[ks] += half;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int h8 = 0; h8 < 2; ++h8) tr_cur[db][h8] += half;
  }
#pragma unroll
  for (int j = 0; j < BWD_LOOK; ++j) win[j] = fetch(j);
  // The loads of tile i + AHEAD go out one at a time between the MFMAs of the pass: issued in one burst
  // after the barrier, they hold up the wave's instruction stream while the memory pipeline takes them in.
  constexpr int LOAD_GAP = NBODY / G::NL;
  // Causal: the tiles a wave's rows see end with the one that holds its last row.  Behind that a wave only takes its share of the loads, and
  // leaves the matrix pipe to the wave beside it (of the 4 tiles on the diagonal of 256 rows, 1.5 on average).
  // (KG = 2: S and dP change registers from pass to pass, and the passes come in pairs; one behind the last tile has every key hidden.)
  const int own_nt = qw0 >= p.Sq ? 0 : (p.causal && qw0 / BWD_ROWS + 1 < nt ? qw0 / BWD_ROWS + 1 : nt) + KG - 1 & ~(KG - 1), all_nt = nt + KG - 1 & ~(KG - 1);
  auto next_pass = [&]() {
    // tile i+1 must have landed before this body reads it (KG = 2: i+2); tile i-1 is free for tile i+AHEAD.  (The operands in flight, one read
    // each, are of tile i+1 or later.)
    __builtin_amdgcn_s_waitcnt(0x0070 | (G::NL & 15) | ((G::NL >> 4) << 14) | (BWD_LOOK << 8));
    barrier_alone();
  };
  auto list_of = [&](int i, int list, f32x16& sc, f32x16& dc, f32x16& sn, f32x16& dn) {
    const int key0 = (2 * i + (KG == 2 ? kg : list)) * 32;  // first key of the half-tile whose dS is formed in this list
    // diagonal: hide the keys after each lane's query; last tile: hide the keys past the end (their K
    // and V rows arrive as zeros, but P = exp(0 - lse) overflows for lse < -88 and inf * 0 is NaN)
    if ((p.causal && key0 + 31 > qw0) || key0 + 31 >= p.Sk) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (key0 + 8 * (v >> 2) + 4 * hh + (v & 3) > lim) sc[v] = hidden;
    }
    if (!MIXED) {
      zero16(sn);
      zero16(dn);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NLIST; ++j) {
      const int J = list * NLIST + j;
      const frag a = win[J % BWD_LOOK];
      win[J % BWD_LOOK] = fetch(J + BWD_LOOK);
      __builtin_amdgcn_sched_barrier(0);
      if (j < NA) {
        const int ks = j >> 1;
        if (MIXED) {
          if (j & 1) {
            if (ks == 0) MA::first_v(dn, a, dof[0]); else MA::acc_v(dn, a, dof[ks]);
          } else {
            if (ks == 0) MA::first_v(sn, a, qf[0]); else MA::acc_v(sn, a, qf[ks]);
          }
        } else if (j & 1) {
          dn = M::run(a, dof[ks], dn);
        } else {
          sn = M::run(a, qf[ks], sn);
        }
        // element-wise work on the current half-tile, spread over the producing MFMAs
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (v * NA / 16 == j) {
            const float pr = fast_exp2(__builtin_fmaf(sc[v], c, -l2));
            sc[v] = pr * (dc[v] - dl);
          }
        if (j == NA / 2 - 1)
          dsf[0] = M::pack(sc[0], sc[1], sc[2], sc[3], sc[4], sc[5], sc[6], sc[7]);
        if (j == NA - 1) dsf[1] = M::pack(sc[8], sc[9], sc[10], sc[11], sc[12], sc[13], sc[14], sc[15]);
      } else {
        const int jb = j - NA;
        const int db = jb % (D / 32), u = jb / (D / 32);
        if (MIXED)
          MA::acc_a(dq[db], a, dsf[u]);
        else
          dq[db] = M::run(a, dsf[u], dq[db]);
      }
      if (J % LOAD_GAP == LOAD_GAP / 2 && J / LOAD_GAP < G::NL) issue_one(i + AHEAD, J / LOAD_GAP);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto pass = [&](int i, f32x16& s0, f32x16& d0, f32x16& s1, f32x16& d1) {
    next_pass();
    if constexpr (KG == 1) set_addresses(i);
    __builtin_amdgcn_sched_barrier(0);
    list_of(i, 0, s0, d0, s1, d1);
    if constexpr (KG == 1) {
      list_of(i, 1, s1, d1, s0, d0);
    } else {
      st_before = st_this;
      st_this = st_next;
      st_next = st_after;
      st_after = st_after == stage_of(G::STAGES - 1) ? stage_of(0) : st_after + G::STAGE;
    }
  };
  for (int i = 0; i < own_nt;) {
    pass(i, sc, dc, sn, dn);
    if constexpr (KG == 2) pass(i + 1, sn, dn, sc, dc);
    i += KG;
    if (i == own_nt) mfma_settle();
  }
  if (own_nt == 0) mfma_settle();  // (a wave without rows)
  for (int i = own_nt; i < all_nt; ++i) {
    next_pass();
    issue_tile(i + AHEAD);
  }
  wait_loads_but<0>();  // nothing may still be writing LDS when the workgroup ends
  // The last MFMAs must have written dq before it is read.  The accumulators are operands of the
  // wait, so no read of them can be scheduled above it.
  if constexpr (MIXED) asm volatile("s_nop 15\n s_nop 15" : "+a"(dq[0]), "+a"(dq[1]), "+a"(dq[2]), "+a"(dq[3])::"memory");

  constexpr int SUMS = D / 32 * 16 * 64;  // (KG = 2) floats of a wave's sums
  if constexpr (KG == 2) {
    __syncthreads();
    float* const sums = (float*)smem + rg * SUMS;
    if (kg == 1) {
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) sums[(db * 16 + v) * 64 + lane] = dq[db][v];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) dq[db][v] += sums[(db * 16 + v) * 64 + lane];
  }

  if (p.grads_in_t) {
    // the whole gradient of the row: written in q's element type, nothing read
    if constexpr (KG == 1) __syncthreads();  // every wave is done with the tiles, and with its loads into them
    T* const dqp = (T*)p.dq + b * p.dqs.b + h * p.dqs.h;
    store_rows<T, D>(dq, p.scale, [&](int r) { return dqp + (int64_t)row_of(qw0 + r) * p.dqs.s; }, p.Sq - qw0, smem + (KG == 2 ? RG * SUMS * 4 : 0) + w * (32 * C::ROWB), lane);
  } else if (qrow < p.Sq) {
    float* dqp = p.dq + b * p.dqs.b + h * p.dqs.h + (int64_t)qrow * p.dqs.s;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4* dst = (f32x4*)(dqp + db * 32 + 8 * g + 4 * hh);
        f32x4 x = *dst;
        x[0] += dq[db][4 * g + 0] * p.scale;
        x[1] += dq[db][4 * g + 1] * p.scale;
        x[2] += dq[db][4 * g + 2] * p.scale;
        x[3] += dq[db][4 * g + 3] * p.scale;
        *dst = x;
      }
  }
}

// ------------------------------------------------------------------------------------------
// dK / dV kernel
// ------------------------------------------------------------------------------------------
template <bool V>
struct Flag {
  static constexpr bool value = V;
};

template <int D>
struct DkvCfg {
  typedef BwdCfg<D> C;
  static constexpr int STAT = 2 * BWD_ROWS * 4;       // lse and delta of the tile's query rows
  static constexpr int STAGE = 2 * C::TILEB + STAT;   // Q tile, dO tile, stats
  static constexpr int SMEM = BWD_STAGES * STAGE + (BWD_THREADS / 64) * 2 * BWD_ROWS * 4;  // (and each wave's copy of two tiles' lse)
  static constexpr int NL = 2 * C::NDMA + 1;          // loads per thread and stage
};

// ASM = false: the D = 128 kernel with every MFMA left to the compiler (its uniform accumulator
// form, its own hazard handling): slower, kept as the test twin of the hand-issued form.
// QG = 2: 64 keys a workgroup.  Its waves come in two groups that own the same keys, and each takes 32 of a tile's 64 query rows; their sums
// are added through LDS.
template <typename T, int D, bool ASM = true, int ADDR = ADDR_PLAIN, int QG = 1>
__global__ void __launch_bounds__(BWD_THREADS, D <= 64 ? 2 : 1) flash_bwd_dkdv_kernel(const BwdParams pk) {
  BwdParams p = pk;  // a variable-length batch rewrites the sizes and bases for its sequence below
  typedef BwdCfg<D> C;
  typedef DkvCfg<D> G;
  typedef Mma16<T> M;
  typedef MmaAsm<T> MA;
  constexpr bool MIXED = D == 128 && ASM;  // see the dq kernel, and MmaAsm
  typedef typename M::frag frag;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  int b, h, kt;
  constexpr int KEYS = 128 / QG;
  if (!workgroup_tile(p, false, KEYS, lane, b, h, kt)) return;
  const int k0 = kt * KEYS;
  const int qg = QG == 2 ? w >> 1 : 0;  // the wave's half of the rows of a tile
  const int kw0 = k0 + (QG == 2 ? w & 1 : w) * 32;
  RowMap map = {};
  select_sequence<T>(p, b, map);
  constexpr bool MAP = ADDR == ADDR_MAP;
  auto row_of = [&](int r) { return MAP ? map.at(r, p.map.pitch) : r; };        // where row r of the sequence lies
  auto stat_of = [&](int r) { return MAP ? map.at(r, p.map.lse_pitch) : r; };   // in lse and delta
  // rows of the tensors from the sequence's first to its last
  const int span_q = MAP ? (p.map.P - 1) * p.map.pitch + p.Sq / p.map.P : p.Sq, span_k = MAP ? span_q : p.Sk;
  if (k0 >= p.Sk || p.Sq <= 0 || (p.causal && k0 >= p.Sq)) {  // no query sees these keys: nothing to add to dk, dv
    if (p.grads_in_t && kw0 + ln < p.Sk) {                     // written gradients of such keys are zero
      zero_grad_row<T, D>((T*)p.dk + b * p.dks.b + h * p.dks.h + (int64_t)row_of(kw0 + ln) * p.dks.s, hh);
      zero_grad_row<T, D>((T*)p.dv + b * p.dvs.b + h * p.dvs.h + (int64_t)row_of(kw0 + ln) * p.dvs.s, hh);
    }
    return;
  }

  const T* qp = (const T*)p.q + b * p.qs.b + h * p.qs.h;
  const T* kp = (const T*)p.k + b * p.ks.b + h * p.ks.h;
  const T* vp = (const T*)p.v + b * p.vs.b + h * p.vs.h;
  const T* dop = (const T*)p.dout + b * p.dos.b + h * p.dos.h;
  const float* lsep = p.lse + ((int64_t)b * p.H + h) * p.lse_bh;
  const float* delp = p.delta + ((int64_t)b * p.H + h) * p.lse_bh;

  const int krow = kw0 + ln;
  frag kf[D / 16], vf[D / 16];
  const float c = p.scale_log2;
  const float hidden = c < 0.f ? INFINITY : -INFINITY;  // a hidden score: exp2(hidden * c - lse) = 0 for either sign of the scale

  // causal: query rows before the first key of this workgroup see none of its keys
  const int it0 = p.causal ? k0 / BWD_ROWS : 0;
  const int nt = (p.Sq + BWD_ROWS - 1) / BWD_ROWS;  // query tiles it0 .. nt-1 are visited

  TileLoader<T, D, BWD_THREADS, ADDR> qld, dold;
  qld.init(qp, p.qs.s, p.Sq, span_q, tid);
  dold.init(dop, p.dos.s, p.Sq, span_q, tid);
  // per-row statistics: waves 0, 2 fetch the tile's 64 lse values, waves 1, 3 its 64 delta values
  // (the pairs store the same bytes to the same place, which keeps every wave's load count equal)
  const u32x4 stat_rsrc = buffer_descriptor((w & 1) ? delp : lsep, (unsigned)(MAP ? (p.map.P - 1) * p.map.lse_pitch + p.Sq / p.map.P : p.Sq) * 4u);
  TileReads<D> rd;
  rd.init(lane);
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_u8*)smem;
  auto stage_of = [&](int i) { return lds0 + (unsigned)((i & (BWD_STAGES - 1)) * G::STAGE); };
  ShardTiles<T, D, BWD_THREADS> tiles;
  if constexpr (MAP) tiles.init(map, it0 * BWD_ROWS);
  auto issue_one = [&](int i, int n) {  // load n of tile i's G::NL (in order): Q, dO and their statistics -> its stage
    const unsigned st = stage_of(i);
    const unsigned dst = st + w * 1024;
    if (n == 2 * C::NDMA) {
      load_to_lds_b32(stat_rsrc, MAP ? tiles.stat_at : i < nt ? (unsigned)(i * BWD_ROWS + lane) * 4u : OFF_NONE, st + 2 * C::TILEB + (w & 1) * (BWD_ROWS * 4));
    } else if constexpr (MAP) {
      if (n == 0) {
        if (QG == 1 || i < nt)
          tiles.find(map, p.map, i * BWD_ROWS, p.Sq, qld, dold, lane, i < nt);
        else
          tiles.repeat_first();
      }
      const int t = n / C::NDMA, q = n % C::NDMA;
      load_to_lds_b128(t ? dold.rsrc : qld.rsrc, tiles.at[t][q], dst + t * C::TILEB + q * (BWD_THREADS * 16));
    } else if (n < C::NDMA) {
      qld.load(n, QG == 2 || i < nt, (QG == 2 && i >= nt ? nt - 1 : i) * BWD_ROWS, dst, map, p.map.pitch);
    } else {
      dold.load(n - C::NDMA, i < nt, i * BWD_ROWS, dst + C::TILEB, map, p.map.pitch);
    }
  };
  auto issue_tile = [&](int i) {
#pragma unroll
    for (int n = 0; n < G::NL; ++n) issue_one(i, n);
  };

  f32x16 dk[D / 32], dv[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    zero16(dk[i]);
    zero16(dv[i]);
  }

  // Half-tile g = 2 i + t is query rows [32 g, 32 g + 32).  Three of them are in work at any time: while the matrix pipe forms S and
  // dP of half g + 1 and the products of half g - 1 or g with the keys' gradients, the vector unit forms P and dS of half g.  The
  // matrix instructions come in groups of GROUP, each with the vector work on 8 of the lane's 16 rows between them: one wave a SIMD issues one
  // instruction every four clocks, and with all vector work beside the MFMAs of S and dP those waited for it and the others for LDS.
  // Bound: matrix pipe and LDS alike (a tile's 64 MFMAs are 2048 clocks; its 112 LDS reads a wave, 4 clocks of the CU's one pipe each whatever
  // their width, and the loads into LDS, 2050).  Causal [1, 32768, 16, 128]: 7.98 -> 7.35 ms.
  //   first group of half g : S, dP of half g + 1, contraction steps 0 .. HS - 1  | P, dS of g, rows 0 .. 7  | dV, dK from g - 1, rows 8 .. 15
  //   second group          : S, dP of half g + 1, steps HS .. 2 HS - 1           | rows 8 .. 15             | dV, dK from g, rows 0 .. 7
  // One pass of the loop runs the second group of half 2 i, both groups of half 2 i + 1 and the first of half 2 i + 2, so that it
  // reads tiles i and i + 1 only.
  // QG = 2: "half g" is the wave's half of tile g; a pass runs the second group of half i and the first of half i + 1, and reads tiles i to i + 2.
  constexpr int HS = D / 32, GROUP = 4 * HS, GROUPS = 4 / QG, NBODY = GROUPS * GROUP;
  constexpr int BWD_LOOK = D <= 64 ? 4 : BWD_LOOK_MAX;  // (two waves per SIMD at D <= 64, as in the dq kernel)
  static_assert(GROUP % BWD_LOOK == 0, "the operand window must tile a group");

  // A wave without keys, or with keys that no query sees, only takes its share of the loads: of a sequence of 16 rows three of four, which held up the
  // fourth at LDS.  Causal, with the masks of halves that need none left out, 16 heads: 2000 sequences of 16 rows 942 -> 881 us, 1000 of 64 546 -> 522,
  // 500 of 128 404 -> 395.
  const bool idle = kw0 >= p.Sk || (p.causal && kw0 >= p.Sq);
  if (it0 < nt) {  // uniform; a workgroup whose keys no query sees adds nothing
    // the workgroup's keys first, as two tiles each of K and V in the stages of tiles it0 + 2 and it0 + 3 (64 keys: both in the last)
    {
      TileLoader<T, D, BWD_THREADS, ADDR> kld, vld;
      kld.init(kp, p.ks.s, p.Sk, span_k, tid);
      vld.init(vp, p.vs.s, p.Sk, span_k, tid);
      const unsigned kdst = stage_of(it0 + 4 - 2 / QG) + w * 1024, vdst = stage_of(it0 + 3) + (QG - 1) * C::TILEB + w * 1024;
#pragma unroll
      for (int half = 0; half < 2 / QG; ++half)
#pragma unroll
        for (int q = 0; q < C::NDMA; ++q) kld.load(q, k0 + half * BWD_ROWS < p.Sk, k0 + half * BWD_ROWS, kdst + half * C::TILEB, map, p.map.pitch);
#pragma unroll
      for (int half = 0; half < 2 / QG; ++half)
#pragma unroll
        for (int q = 0; q < C::NDMA; ++q) vld.load(q, k0 + half * BWD_ROWS < p.Sk, k0 + half * BWD_ROWS, vdst + half * C::TILEB, map, p.map.pitch);
    }
    issue_tile(it0);
    if constexpr (QG == 1) {
      wait_loads_but<G::NL>();
      __syncthreads();
      const unsigned own = (w >> 1) * C::TILEB + (w & 1) * 32 * C::ROWB;  // the wave's 32 keys in either pair of tiles
      read_rows<frag, D>(kf, stage_of(it0 + 2) + own, rd);
      read_rows<frag, D>(vf, stage_of(it0 + 3) + own, rd);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage of tile it0 + 2 has been read ...
      issue_tile(it0 + 1);
      __syncthreads();                     // ... by every wave
      issue_tile(it0 + 2);
      wait_loads_but<2 * G::NL>();
      __syncthreads();
    } else {
      issue_tile(it0 + 1);
      issue_tile(it0 + 2);
      wait_loads_but<G::NL>();
      __syncthreads();
      const unsigned own = stage_of(it0 + 3) + (w & 1) * 32 * C::ROWB;
      read_rows<frag, D>(kf, own, rd);
      read_rows<frag, D>(vf, own + C::TILEB, rd);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): read, before the barrier of the first pass
    }

  }
  if (it0 < nt && idle) {
    // its share of the loads, and the barriers of the passes (of which there is an even number with QG = 2)
    for (int i = it0, end = QG == 1 ? nt : it0 + (nt - it0 + 1 & ~1); i < end; ++i) {
      wait_loads_but<QG == 2 ? 0 : G::NL>();
      barrier_alone();
      issue_tile(i + 3);
    }
    wait_loads_but<0>();
  }
  if (it0 < nt && !idle) {
    // V negated: with delta as the accumulator's start the products give delta - dP, and -dS costs one multiplication per element.
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      u32x4 x = __builtin_bit_cast(u32x4, vf[ks]);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] ^= 0x80008000u;
      vf[ks] = as_frag<frag>(x);
    }

    // Per-lane LDS addresses of the operands; each is moved on to the next tile where that tile is first read through it.
    unsigned row_at[D / 16], tr_at[D / 32][2], stat_at = stage_of(it0) + 2 * C::TILEB + 16 * hh;
    unsigned step = 0, last_step = 0, next_step = 0;  // from tile i to i + 1, from i - 1 to i, from i + 1 to i + 2
    const unsigned half = qg * 32 * C::ROWB;          // (QG = 2) the wave's half of a tile
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) row_at[ks] = stage_of(it0) + half + rd.row[ks];
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int h8 = 0; h8 < 2; ++h8) tr_at[db][h8] = stage_of(it0) + half + rd.tr[db][h8];
    auto advance = [&](unsigned& at, unsigned by) {
      at += by;
      asm volatile("" : "+v"(at));  // (kept, not formed again from the tile's number at every use)
    };

    f32x16 s0, d0, s1, d1;  // S and delta - dP of the current and the next half-tile, in turn
    frag pf[2], dsf[2];
    u32x4 pw, dsw;
    f32x4 ln_next[2], ln_cur[2];  // -lse log2 e of the 8 rows of the next / the current group
    // The wave's own copy of a tile's lse, times -log2 e: a lane prepares one row (a lane works on 16 of each half-tile).
    typedef __attribute__((address_space(3))) float lds_float;
    const unsigned own_lse = lds0 + BWD_STAGES * G::STAGE + w * (2 * BWD_ROWS * 4);
    auto lse_of = [&](int i) { return own_lse + (unsigned)((i & 1) * (BWD_ROWS * 4)); };
    float lse_row;
    auto read_lse_row = [&](unsigned stage) { lse_row = *(const lds_float*)(lds_u8*)(uintptr_t)(stage + 2 * C::TILEB + 4 * lane); };
    // (QG = 2, behind the last tile: P = 0 for its rows, which are the last tile's of Q; rows of zeros would give NaN where a key holds an infinity)
    auto write_lse_row = [&](int i) {
      *(lds_float*)(lds_u8*)(uintptr_t)(lse_of(i) + 4 * lane) = QG == 1 || i < nt ? lse_row * -1.4426950408889634f : -INFINITY;
    };
    auto load_lse = [&](f32x4 (&l)[2], unsigned at, int row) {
#pragma unroll
      for (int g = 0; g < 2; ++g) l[g] = __builtin_bit_cast(f32x4, lds_read_b128(at + 16 * hh + (row + 8 * g) * 4));
    };
    auto load_delta = [&](f32x16& x, unsigned at, int row) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 d4 = __builtin_bit_cast(f32x4, lds_read_b128(at + (BWD_ROWS + row + 8 * g) * 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * g + e] = d4[e];
      }
    };
    // diagonal: a key sees only the queries at or after it
    auto mask = [&](f32x16& sc, int half) {
      const int r0 = half * 32;
      if (kw0 + 31 <= r0) return;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (krow > r0 + 8 * (v >> 2) + 4 * hh + (v & 3)) sc[v] = hidden;
    };
    // part n of the vector work of a group on rows 8 u .. 8 u + 7 of the lane's 16: two parts per row
    // (pinned by the empty asm: left alone, the compiler moves all of it behind the next branch)
    float pr[8], ds[8];
    auto element = [&](const f32x16& sc, const f32x16& dc, int u, int n) {
      const int e = n >> 1, v = 8 * u + e;
      if ((n & 1) == 0) {
        pr[e] = fast_exp2(__builtin_fmaf(sc[v], c, ln_cur[e >> 2][e & 3]));
        asm volatile("" : "+v"(pr[e]));
      } else {
        ds[e] = dc[v] * pr[e];
        asm volatile("" : "+v"(ds[e]));
        if (e & 1) {
          pw[e >> 1] = M::pack2(pr[e - 1], pr[e]);
          dsw[e >> 1] = M::pack2(ds[e - 1], ds[e]);
        }
        if (e == 7) {
          pf[u] = as_frag<frag>(pw);
          dsf[u] = as_frag<frag>(dsw);
          asm volatile("" : "+v"(pf[u]), "+v"(dsf[u]));
        }
      }
    };
    auto mma_s = [&](f32x16& x, frag a, int ks) {
      if (!MIXED) {
        if (ks == 0) zero16(x);
        x = M::run(a, kf[ks], x);
      } else if (ks == 0) {
        MA::first_v(x, a, kf[0]);
      } else {
        MA::acc_v(x, a, kf[ks]);
      }
    };
    auto mma_d = [&](f32x16& x, frag a, int ks) {
      if (MIXED)
        MA::acc_v(x, a, vf[ks]);
      else
        x = M::run(a, vf[ks], x);
    };

    // Matrix instruction n of a group: 0 .. KS - 1: S, contraction step; KS .. : dP; 2 KS ..: gradient product number.  The gradient
    // products, whose operands take twice as many LDS reads, are every other one.
    constexpr int KS = D / 16;
    auto instruction = [](bool first, int n) -> int {
      const int k = n >> 1;
      return (n & 1) ? 2 * KS + k : (first ? 0 : HS) + (k < HS ? k : KS + k - HS);
    };
    // The first vector instruction that reads S is the mask in front of the next group, the first that reads dP part 1 of element(), behind the
    // second matrix instruction of that group: nine of them come after the last of S and three after the last of dP.
    constexpr int LAST_S = 2 * HS - 2, LAST_DP = 4 * HS - 2;
    static_assert(instruction(false, LAST_S) == KS - 1 && instruction(false, LAST_DP) == 2 * KS - 1, "the last of S and of dP");
    static_assert(!MIXED || (GROUP == 16 && GROUP - 1 - LAST_S >= MFMA_APART && GROUP - 1 - LAST_DP + 2 >= MFMA_APART), "distance to the element-wise work");
    // operand number J of the pass on tile i (J >= NBODY: the first operands of the next pass)
    auto fetch = [&](int J) -> frag {
      const int group = J % NBODY / GROUP;
      const int n = instruction(group & 1, J % GROUP);
      if (n < 2 * KS) {  // row of Q (S) or dO (dP) of the half-tile being produced
        const int ks = n % KS, which = n / KS;
        if constexpr (QG == 2) {
          if (which == 0) advance(row_at[ks], group == 1 || J >= NBODY ? next_step : step);
          return as_frag<frag>(lds_read_b128(row_at[ks] + which * C::TILEB));
        }
        if ((group == 1 || group == 2) && which == 0) advance(row_at[ks], step);
        return as_frag<frag>(lds_read_b128(row_at[ks] + (group == 1 || group == 2 ? 0 : 32 * C::ROWB) + which * C::TILEB));
      }
      // jb = db * 2 + which: dO^T (for dV) or Q^T (for dK) of the 16 rows whose P and dS are used
      const int jb = n - 2 * KS, which = jb & 1, db = jb >> 1;
      if (group == 0 && which == 0) {
#pragma unroll
        for (int h8 = 0; h8 < 2; ++h8) advance(tr_at[db][h8], J >= NBODY ? step : last_step);
      }
      const unsigned off = (which ? 0 : C::TILEB) + 16 * group * C::ROWB;
      return frag_tr<frag>(tr_at[db][0] + off, tr_at[db][1] + off);
    };

    // Before the loop: S, dP of half 0 and what the first group of half 0 would do, less the gradients of a half before it.
    read_lse_row(stage_of(it0));
    write_lse_row(it0);
    load_lse(ln_cur, lse_of(it0), 32 * qg);
    load_lse(ln_next, lse_of(it0), 32 * qg + 16);
    load_delta(d0, stat_at, 32 * qg);
    if constexpr (QG == 2) {
      read_lse_row(stage_of(it0 + 1));
      write_lse_row(it0 + 1);
      stat_at += stage_of(it0 + 1) - stage_of(it0);
      load_delta(d1, stat_at, 32 * qg);
    } else {
      load_delta(d1, stat_at, 32);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      mma_s(s0, as_frag<frag>(lds_read_b128(row_at[ks])), ks);
      mma_d(d0, as_frag<frag>(lds_read_b128(row_at[ks] + C::TILEB)), ks);
    }
#pragma unroll
    for (int ks = 0; ks < HS; ++ks) {
      if (QG == 2) row_at[ks] += stage_of(it0 + 1) - stage_of(it0);
      mma_s(s1, as_frag<frag>(lds_read_b128(row_at[ks] + (QG == 2 ? 0 : 32 * C::ROWB))), ks);
      mma_d(d1, as_frag<frag>(lds_read_b128(row_at[ks] + (QG == 2 ? 0 : 32 * C::ROWB) + C::TILEB)), ks);
    }
    frag win[BWD_LOOK];
    if (QG == 2) step = stage_of(it0 + 1) - stage_of(it0);
#pragma unroll
    for (int j = 0; j < BWD_LOOK; ++j) win[j] = fetch(j);
    if (QG == 2) step = 0;
    if (MIXED) mfma_settle();
    if (p.causal) mask(s0, 2 * it0 + qg);
#pragma unroll
    for (int n = 0; n < 16; ++n) element(s0, d0, 0, n);

    // The loads of tile i + 3 go out one at a time between the MFMAs of the pass: issued in one
    // burst after the barrier, they hold up the wave's instruction stream while the memory pipeline
    // takes them in.
    constexpr int LOAD_GAP = QG == 2 ? 2 : NBODY / G::NL;
    static_assert(LOAD_GAP / 2 + (G::NL - 1) * LOAD_GAP < NBODY, "all loads of a tile in one pass");
    // half-tiles in work at the start: s0, d0 (vector work) and s1, d1 (in production)
    auto pass = [&](int i, f32x16& s0, f32x16& d0, f32x16& s1, f32x16& d1, auto diagonal) {
      // tile i + 1 has landed (QG = 2: i + 2, requested in the pass before); every wave is done with tile i - 1.  The operands in flight are of
      // later tiles, so nothing else is waited for.
      wait_loads_but<QG == 2 ? 0 : G::NL>();
      if (MIXED)
        barrier_alone();
      else
        __syncthreads();
      last_step = step;
      step = stage_of(i + 1) - stage_of(i);
      next_step = stage_of(i + 2) - stage_of(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int group = 0; group < GROUPS; ++group) {
        f32x16 &sc = group == 1 || group == 2 ? s1 : s0, &dc = group == 1 || group == 2 ? d1 : d0;  // half-tile of the vector work
        f32x16 &sn = group == 1 || group == 2 ? s0 : s1, &dn = group == 1 || group == 2 ? d0 : d1;
        if (diagonal.value && (group & 1)) mask(sc, 2 * i + (group + 1) / 2);
        ln_cur[0] = ln_next[0];
        ln_cur[1] = ln_next[1];
        // a row of lse for the wave's copy; the next group's lse rows; what dP of the half-tile in production starts from
        if (group == 0) read_lse_row(stage_of(i + QG));
        if (group == 1) write_lse_row(i + QG);
        if constexpr (QG == 2) {
          if (group == 1) {
            stat_at += next_step;
            load_delta(dn, stat_at, 32 * qg);
          }
          load_lse(ln_next, lse_of(i + 1), 32 * qg + 16 * group);
        } else {
          if (group == 2) stat_at += step;
          if (group & 1) load_delta(dn, group == 1 ? stat_at + step : stat_at, group == 1 ? 0 : 32);
          load_lse(ln_next, lse_of(group < 2 ? i : i + 1), group == 0 ? 32 : group == 1 ? 48 : group == 2 ? 0 : 16);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < GROUP; ++m) {
          const int J = group * GROUP + m;
          const frag a = win[J % BWD_LOOK];
          win[J % BWD_LOOK] = fetch(J + BWD_LOOK);
          __builtin_amdgcn_sched_barrier(0);
          const int n = instruction(group & 1, m);
          if (n < KS) {
            mma_s(sn, a, n);
          } else if (n < 2 * KS) {
            mma_d(dn, a, n - KS);
          } else {
            const int jb = n - 2 * KS, which = jb & 1, db = jb >> 1, u = group & 1;
            if (!MIXED) {
              if (which)
                dk[db] = M::run(a, dsf[u], dk[db]);
              else
                dv[db] = M::run(a, pf[u], dv[db]);
            } else if (which) {
              MA::acc_a(dk[db], a, dsf[u]);
            } else {
              MA::acc_a(dv[db], a, pf[u]);
            }
          }
          // rows 8 .. 15 in the second group of a half-tile, 0 .. 7 in the first
#pragma unroll
          for (int e = m * 16 / GROUP; e < (m + 1) * 16 / GROUP; ++e) element(sc, dc, group & 1 ? 0 : 1, e);
          if (J % LOAD_GAP == LOAD_GAP / 2 && J / LOAD_GAP < G::NL) issue_one(i + 3, J / LOAD_GAP);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    int i = it0;
    if constexpr (QG == 1) {
      // The halves on the diagonal of 128 keys are of tiles it0 and it0 + 1; a loop of their own, as the others would copy S for the choice.
      for (const int end = p.causal ? (it0 + 2 < nt ? it0 + 2 : nt) : it0; i < end; ++i) pass(i, s0, d0, s1, d1, Flag<true>());
      for (; i < nt; ++i) pass(i, s0, d0, s1, d1, Flag<false>());
    } else {
      // The diagonal of 64 keys is in tile it0, whose S has been seen to.  Passes in pairs, as S and dP change registers from one to the next
      // (a pass behind the last tile adds zeros: see write_lse_row; left out, the accumulators are copied where the loop has two ends).
      for (; i < nt; i += 2) {
        pass(i, s0, d0, s1, d1, Flag<false>());
        pass(i + 1, s1, d1, s0, d0, Flag<false>());
      }
    }
    mfma_settle();
    wait_loads_but<0>();
  }
  // The last MFMAs must have written dk / dv before they are read; the accumulators are operands of
  // the wait, so no read of them can be scheduled above it.
  if constexpr (MIXED)
    asm volatile("s_nop 15\n s_nop 15"
                 : "+a"(dk[0]), "+a"(dk[1]), "+a"(dk[2]), "+a"(dk[3]), "+a"(dv[0]), "+a"(dv[1]), "+a"(dv[2]), "+a"(dv[3])::"memory");

  const float dk_scale = -p.scale;  // (-dS, see the loop)
  constexpr int SUMS = D / 32 * 16 * 64;  // (QG = 2) floats of one gradient of a wave
  if constexpr (QG == 2) {
    // group 0 writes dv, group 1 dk: each leaves the other's part in LDS
    __syncthreads();
    float* const own = (float*)smem + w * SUMS;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) own[(db * 16 + v) * 64 + lane] = qg ? dv[db][v] : dk[db][v];
    __syncthreads();
    const float* const other = (const float*)smem + (w ^ 2) * SUMS;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float x = other[(db * 16 + v) * 64 + lane];
        if (qg)
          dk[db][v] += x;
        else
          dv[db][v] += x;
      }
    T* const dst = qg ? (T*)p.dk + b * p.dks.b + h * p.dks.h : (T*)p.dv + b * p.dvs.b + h * p.dvs.h;
    float* const dst32 = qg ? p.dk + b * p.dks.b + h * p.dks.h : p.dv + b * p.dvs.b + h * p.dvs.h;
    const int64_t stride = qg ? p.dks.s : p.dvs.s;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) dv[db][v] = qg ? dk[db][v] * dk_scale : dv[db][v];
    if (p.grads_in_t) {
      store_rows<T, D>(dv, 1.f, [&](int r) { return dst + (int64_t)row_of(kw0 + r) * stride; }, p.Sk - kw0, smem + 4 * SUMS * 4 + w * (32 * C::ROWB), lane);
    } else if (krow < p.Sk) {
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4* const to = (f32x4*)(dst32 + (int64_t)krow * stride + db * 32 + 8 * g + 4 * hh);
          f32x4 x = *to;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] += dv[db][4 * g + e];
          *to = x;
        }
    }
    return;
  }
  if (p.grads_in_t) {
    __syncthreads();  // every wave is done with the tiles, and with its loads into them
    T* const dkp = (T*)p.dk + b * p.dks.b + h * p.dks.h;
    T* const dvp = (T*)p.dv + b * p.dvs.b + h * p.dvs.h;
    store_rows<T, D>(dv, 1.f, [&](int r) { return dvp + (int64_t)row_of(kw0 + r) * p.dvs.s; }, p.Sk - kw0, smem + w * (64 * C::ROWB), lane);
    store_rows<T, D>(dk, dk_scale, [&](int r) { return dkp + (int64_t)row_of(kw0 + r) * p.dks.s; }, p.Sk - kw0, smem + w * (64 * C::ROWB) + 32 * C::ROWB, lane);
  } else if (krow < p.Sk) {
    float* dkp = p.dk + b * p.dks.b + h * p.dks.h + (int64_t)krow * p.dks.s;
    float* dvp = p.dv + b * p.dvs.b + h * p.dvs.h + (int64_t)krow * p.dvs.s;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4* d1 = (f32x4*)(dkp + db * 32 + 8 * g + 4 * hh);
        f32x4* d2 = (f32x4*)(dvp + db * 32 + 8 * g + 4 * hh);
        f32x4 x = *d1, y = *d2;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] += dk[db][4 * g + e] * dk_scale;
          y[e] += dv[db][4 * g + e];
        }
        *d1 = x;
        *d2 = y;
      }
  }
}

// ------------------------------------------------------------------------------------------
// fp32 kernels: the same two-kernel scheme on v_mfma_f32_32x32x2_f32 (fp32 products and
// accumulation, P and dS stay fp32).  Correctness path for fp32 inputs: tiles of 32 rows staged
// through registers, no software pipeline.  The contraction index of the gradient products is the
// row an accumulator register holds (8*(v/4) + 4*hh + v%4), so P and dS are used where they are.
// Bound: the chain of a wave, 192 (dq) or 256 (dk / dv) matrix instructions of 64 clocks per tile at D = 128, while the grid is small.
// SHARED: a workgroup owns 32 rows (keys) and its four waves take every fourth tile, each through LDS of its own (the next
// tile waits in registers, no barrier in the loop), and their sums are combined through LDS at the end: a quarter of the chain.
// Backward, causal: [1, 288, 16, 128] 172 -> 79 us, [1, 1000, 12, 64] 318 -> 108, [1, 2048, 16, 128] 1081 -> 690.
// ------------------------------------------------------------------------------------------
constexpr int B32_ROWS = 32;
constexpr int B32_WAVES = BWD_THREADS / 64;

template <int D>
struct Bwd32Cfg {
  static constexpr int PITCH = D + 4;              // floats per LDS row
  static constexpr int TILE = B32_ROWS * PITCH;    // floats per tile
  static constexpr int STAT = 2 * B32_ROWS;        // lse * log2 e and delta of a query tile
  static constexpr int SMEM_DQ = 2 * 2 * TILE * 4;
  static constexpr int SMEM_DKV = 2 * (2 * TILE + STAT) * 4;
  static constexpr int SMEM_SHARED = B32_WAVES * (2 * TILE + STAT) * 4;  // a pair of tiles per wave; later its sums, 64 D floats
  static constexpr int CPR = D / 4;
};

// two row-major tiles of 32 rows (a, b) of tensors with the same row count, staged together by THREADS threads
template <int D, int THREADS>
struct PairStage {
  typedef Bwd32Cfg<D> C;
  static constexpr int RPP = THREADS / C::CPR;
  static constexpr int PASS = (B32_ROWS + RPP - 1) / RPP;
  f32x4 ra[PASS], rb[PASS];
  template <typename Row>
  __device__ __forceinline__ void gload(const float* a, int64_t as, const float* b, int64_t bs, int row0, int nrows, int tid, Row&& row_of) {
    const int cc = tid % C::CPR, cr = tid / C::CPR;
#pragma unroll
    for (int i = 0; i < PASS; ++i) {
      const int lr = cr + i * RPP;
      if (lr < B32_ROWS) {
        int r = row0 + lr;
        r = row_of(r < nrows ? r : nrows - 1);
        ra[i] = *(const f32x4*)(a + (int64_t)r * as + cc * 4);
        rb[i] = *(const f32x4*)(b + (int64_t)r * bs + cc * 4);
      }
    }
  }
  __device__ __forceinline__ void lstore(float* ta, float* tb, int tid) const {
    const int cc = tid % C::CPR, cr = tid / C::CPR;
#pragma unroll
    for (int i = 0; i < PASS; ++i) {
      const int lr = cr + i * RPP;
      if (lr < B32_ROWS) {
        *(f32x4*)(ta + lr * C::PITCH + cc * 4) = ra[i];
        *(f32x4*)(tb + lr * C::PITCH + cc * 4) = rb[i];
      }
    }
  }
};

// SHARED: a wave's tile goes from registers to the wave's own LDS; its lanes' earlier reads come before, their later ones after.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// The sums of block db, over the waves' records of `floats` floats each.
__device__ __forceinline__ f32x16 sum_records(const float* sm, int floats, int db, int lane) {
  f32x16 x;
  zero16(x);
#pragma unroll
  for (int j = 0; j < B32_WAVES; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) x[v] += sm[j * floats + (db * 16 + v) * 64 + lane];
  return x;
}

template <int D, bool SHARED>
__global__ void __launch_bounds__(BWD_THREADS, 1) flash_bwd32_dq_kernel(const BwdParams pk) {
  BwdParams p = pk;  // a variable-length batch rewrites the sizes and bases for its sequence below
  typedef Bwd32Cfg<D> C;
  extern __shared__ __align__(16) unsigned char smem[];
  float* sm = (float*)smem;
  constexpr int ROWS = SHARED ? 32 : 128;
  const int tid = threadIdx.x;
  const int lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  int b, h, qt;
  if (!workgroup_tile(p, true, ROWS, lane, b, h, qt)) return;
  const int q0 = qt * ROWS;
  const int qw0 = SHARED ? q0 : q0 + w * 32;
  RowMap map = {};
  select_sequence<float>(p, b, map);
  auto row_of = [&](int r) { return p.map.P ? map.at(r, p.map.pitch) : r; };        // where row r of the sequence lies
  auto stat_of = [&](int r) { return p.map.P ? map.at(r, p.map.lse_pitch) : r; };   // in lse and delta
  if (q0 >= p.Sq || p.Sk <= 0) {  // (variable-length batches only) no keys: nothing to add to dq, a written dq is zero
    if (p.grads_in_t && qw0 + ln < p.Sq)
      zero_grad_row<float, D>(p.dq + b * p.dqs.b + h * p.dqs.h + (int64_t)row_of(qw0 + ln) * p.dqs.s, hh);
    return;
  }

  const float* qp = (const float*)p.q + b * p.qs.b + h * p.qs.h;
  const float* kp = (const float*)p.k + b * p.ks.b + h * p.ks.h;
  const float* vp = (const float*)p.v + b * p.vs.b + h * p.vs.h;
  const float* dop = (const float*)p.dout + b * p.dos.b + h * p.dos.h;

  const int qrow = qw0 + ln;
  const int qrow_c = qrow < p.Sq ? qrow : p.Sq - 1;
  // contraction step of the first products: head dim 8*g + 4*hh + e
  f32x4 qf[D / 8], dof[D / 8];
#pragma unroll
  for (int g = 0; g < D / 8; ++g) {
    qf[g] = *(const f32x4*)(qp + (int64_t)row_of(qrow_c) * p.qs.s + 8 * g + 4 * hh);
    dof[g] = *(const f32x4*)(dop + (int64_t)row_of(qrow_c) * p.dos.s + 8 * g + 4 * hh);
  }
  const int64_t li = ((int64_t)b * p.H + h) * p.lse_bh + stat_of(qrow_c);
  const float l2 = p.lse[li] * 1.4426950408889634f;
  float dl;
  if (p.out) {  // delta = rowsum(dout * out), written for the dk / dv kernel
    const float* op = (const float*)p.out + b * p.os.b + h * p.os.h + (int64_t)row_of(qrow_c) * p.os.s;
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < D / 8; ++g) {
      const f32x4 x = *(const f32x4*)(op + 8 * g + 4 * hh);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = __builtin_fmaf(x[e], dof[g][e], sum);
    }
    dl = halves_sum(sum);
    if (hh == 0 && qrow < p.Sq && (!SHARED || w == 0)) p.delta[li] = dl;
  } else {
    dl = p.delta[li];
  }
  const float c = p.scale_log2;
  const int lim = p.causal ? (qrow < p.Sk - 1 ? qrow : p.Sk - 1) : p.Sk - 1;  // last visible key

  const int kv_end = p.causal ? (q0 + ROWS < p.Sk ? q0 + ROWS : p.Sk) : p.Sk;
  const int nt = (kv_end + B32_ROWS - 1) / B32_ROWS;

  f32x16 dq[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) zero16(dq[i]);

  constexpr int STEP = SHARED ? B32_WAVES : 1, RECORD = 2 * C::TILE + C::STAT;
  const int st_id = SHARED ? lane : tid, first = SHARED ? w : 0;
  float* const own = sm + w * RECORD;  // (SHARED)
  PairStage<D, SHARED ? 64 : BWD_THREADS> st;
  if (first < nt) {
    st.gload(kp, p.ks.s, vp, p.vs.s, first * B32_ROWS, p.Sk, st_id, row_of);
    st.lstore(SHARED ? own : sm, (SHARED ? own : sm) + C::TILE, st_id);
  }
  if (SHARED)
    wave_fence();
  else
    __syncthreads();

  for (int it = first; it < nt; it += STEP) {
    const int cur = it & 1;
    const int key0 = it * B32_ROWS;
    const bool more = it + STEP < nt;
    if (more) st.gload(kp, p.ks.s, vp, p.vs.s, key0 + STEP * B32_ROWS, p.Sk, st_id, row_of);
    if (!(p.causal && key0 > qw0 + 31)) {
      const float* kb = SHARED ? own : sm + cur * 2 * C::TILE;
      const float* vb = kb + C::TILE;
      f32x16 s, dp;
      zero16(s);
      zero16(dp);
#pragma unroll
      for (int g = 0; g < D / 8; ++g) {
        const f32x4 a = *(const f32x4*)(kb + ln * C::PITCH + 8 * g + 4 * hh);
        const f32x4 a2 = *(const f32x4*)(vb + ln * C::PITCH + 8 * g + 4 * hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], qf[g][e], s, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[e], dof[g][e], dp, 0, 0, 0);
        }
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int key = key0 + 8 * (v >> 2) + 4 * hh + (v & 3);
        const float pr = key > lim ? 0.f : fast_exp2(__builtin_fmaf(s[v], c, -l2));
        s[v] = pr * (dp[v] - dl);
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int kl = 8 * (v >> 2) + 4 * hh + (v & 3);
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          dq[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(kb[kl * C::PITCH + db * 32 + ln], s[v], dq[db], 0, 0, 0);
      }
    }
    if constexpr (SHARED) {
      wave_fence();
      if (more) st.lstore(own, own + C::TILE, st_id);
      wave_fence();
    } else {
      if (more) st.lstore(sm + (cur ^ 1) * 2 * C::TILE, sm + (cur ^ 1) * 2 * C::TILE + C::TILE, tid);
      __syncthreads();
    }
    if (SHARED && !more) mfma_settle();
  }

  float* const dqp = p.dq + b * p.dqs.b + h * p.dqs.h + (int64_t)row_of(qrow_c) * p.dqs.s;
  auto store = [&](int db, const f32x16& sum) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4* dst = (f32x4*)(dqp + db * 32 + 8 * g + 4 * hh);
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (!p.grads_in_t) x = *dst;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] += sum[4 * g + e] * p.scale;
      *dst = x;
    }
  };
  if constexpr (SHARED) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) own[(db * 16 + v) * 64 + lane] = dq[db][v];
    __syncthreads();
    for (int db = w; db < D / 32; db += B32_WAVES) {
      const f32x16 sum = sum_records(sm, RECORD, db, lane);
      if (qrow < p.Sq) store(db, sum);
    }
  } else if (qrow < p.Sq) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db) store(db, dq[db]);
  }
}


template <int D, bool SHARED>
__global__ void __launch_bounds__(BWD_THREADS, 1) flash_bwd32_dkdv_kernel(const BwdParams pk) {
  BwdParams p = pk;  // a variable-length batch rewrites the sizes and bases for its sequence below
  typedef Bwd32Cfg<D> C;
  extern __shared__ __align__(16) unsigned char smem[];
  float* sm = (float*)smem;
  constexpr int ROWS = SHARED ? 32 : 128;
  const int tid = threadIdx.x;
  const int lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  int b, h, kt;
  if (!workgroup_tile(p, false, ROWS, lane, b, h, kt)) return;
  const int k0 = kt * ROWS;
  const int kw0 = SHARED ? k0 : k0 + w * 32;
  RowMap map = {};
  select_sequence<float>(p, b, map);
  auto row_of = [&](int r) { return p.map.P ? map.at(r, p.map.pitch) : r; };        // where row r of the sequence lies
  auto stat_of = [&](int r) { return p.map.P ? map.at(r, p.map.lse_pitch) : r; };   // in lse and delta
  if (k0 >= p.Sk || p.Sq <= 0 || (p.causal && k0 >= p.Sq)) {  // no query sees these keys: nothing to add to dk, dv
    if (p.grads_in_t && kw0 + ln < p.Sk) {                     // written gradients of such keys are zero
      zero_grad_row<float, D>(p.dk + b * p.dks.b + h * p.dks.h + (int64_t)row_of(kw0 + ln) * p.dks.s, hh);
      zero_grad_row<float, D>(p.dv + b * p.dvs.b + h * p.dvs.h + (int64_t)row_of(kw0 + ln) * p.dvs.s, hh);
    }
    return;
  }

  const float* qp = (const float*)p.q + b * p.qs.b + h * p.qs.h;
  const float* kp = (const float*)p.k + b * p.ks.b + h * p.ks.h;
  const float* vp = (const float*)p.v + b * p.vs.b + h * p.vs.h;
  const float* dop = (const float*)p.dout + b * p.dos.b + h * p.dos.h;
  const float* lsep = p.lse + ((int64_t)b * p.H + h) * p.lse_bh;
  const float* delp = p.delta + ((int64_t)b * p.H + h) * p.lse_bh;

  const int krow = kw0 + ln;
  const int krow_c = krow < p.Sk ? krow : p.Sk - 1;
  f32x4 kf[D / 8], vf[D / 8];
#pragma unroll
  for (int g = 0; g < D / 8; ++g) {
    kf[g] = *(const f32x4*)(kp + (int64_t)row_of(krow_c) * p.ks.s + 8 * g + 4 * hh);
    vf[g] = *(const f32x4*)(vp + (int64_t)row_of(krow_c) * p.vs.s + 8 * g + 4 * hh);
  }
  const float c = p.scale_log2;

  const int it0 = p.causal ? k0 / B32_ROWS : 0;  // earlier query rows see none of these keys
  const int nt = (p.Sq + B32_ROWS - 1) / B32_ROWS;
  constexpr int STAGE = 2 * C::TILE + C::STAT;

  f32x16 dk[D / 32], dv[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    zero16(dk[i]);
    zero16(dv[i]);
  }

  constexpr int STEP = SHARED ? B32_WAVES : 1;
  const int st_id = SHARED ? lane : tid, first = SHARED ? it0 + w : it0;
  PairStage<D, SHARED ? 64 : BWD_THREADS> st;
  float st_l = 0.f, st_d = 0.f;
  constexpr bool LATE = SHARED && D == 128;  // no registers left for the next pair of tiles: loaded when its place is free
  auto gload = [&](int it) {
    if (!LATE) st.gload(qp, p.qs.s, dop, p.dos.s, it * B32_ROWS, p.Sq, st_id, row_of);
    if (st_id < B32_ROWS) {
      int r = it * B32_ROWS + st_id;
      r = r < p.Sq ? r : p.Sq - 1;
      st_l = lsep[stat_of(r)] * 1.4426950408889634f;
      st_d = delp[stat_of(r)];
    }
  };
  auto lstore = [&](int stage, int it) {
    float* sb = sm + stage * STAGE;
    if (LATE) st.gload(qp, p.qs.s, dop, p.dos.s, it * B32_ROWS, p.Sq, st_id, row_of);
    st.lstore(sb, sb + C::TILE, st_id);
    if (st_id < B32_ROWS) {
      sb[2 * C::TILE + st_id] = st_l;
      sb[2 * C::TILE + B32_ROWS + st_id] = st_d;
    }
  };

  // (stage: SHARED, the wave's own; else two in turn)
  if (first < nt) {
    gload(first);
    lstore(SHARED ? w : first & 1, first);
  }
  if (SHARED)
    wave_fence();
  else
    __syncthreads();

  for (int it = first; it < nt; it += STEP) {
    const int cur = SHARED ? w : it & 1;
    const int r0 = it * B32_ROWS;
    const bool more = it + STEP < nt;
    if (more) gload(it + STEP);
    if (!(p.causal && r0 + B32_ROWS - 1 < kw0)) {
      const float* qb = sm + cur * STAGE;
      const float* dob = qb + C::TILE;
      const float* stp = dob + C::TILE;
      f32x16 s, dp;
      zero16(s);
      zero16(dp);
#pragma unroll
      for (int g = 0; g < D / 8; ++g) {
        const f32x4 a = *(const f32x4*)(qb + ln * C::PITCH + 8 * g + 4 * hh);
        const f32x4 a2 = *(const f32x4*)(dob + ln * C::PITCH + 8 * g + 4 * hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], kf[g][e], s, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[e], vf[g][e], dp, 0, 0, 0);
        }
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ql = 8 * (v >> 2) + 4 * hh + (v & 3);
        const int qi = r0 + ql;
        const bool dead = qi >= p.Sq || (p.causal && krow > qi);
        const float pr = dead ? 0.f : fast_exp2(__builtin_fmaf(s[v], c, -stp[ql]));
        s[v] = pr;
        dp[v] = pr * (dp[v] - stp[B32_ROWS + ql]);
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ql = 8 * (v >> 2) + 4 * hh + (v & 3);
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
          dv[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(dob[ql * C::PITCH + db * 32 + ln], s[v], dv[db], 0, 0, 0);
          dk[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(qb[ql * C::PITCH + db * 32 + ln], dp[v], dk[db], 0, 0, 0);
        }
      }
    }
    if constexpr (SHARED) {
      wave_fence();
      if (more) lstore(w, it + STEP);
      wave_fence();
    } else {
      if (more) lstore(cur ^ 1, it + 1);
      __syncthreads();
    }
    if (!more) mfma_settle();
  }

  float* const dkp = p.dk + b * p.dks.b + h * p.dks.h + (int64_t)row_of(krow_c) * p.dks.s;
  float* const dvp = p.dv + b * p.dvs.b + h * p.dvs.h + (int64_t)row_of(krow_c) * p.dvs.s;
  auto store = [&](float* to, int db, const f32x16& sum, float scale) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4* dst = (f32x4*)(to + db * 32 + 8 * g + 4 * hh);
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (!p.grads_in_t) x = *dst;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] += sum[4 * g + e] * scale;
      *dst = x;
    }
  };
  if constexpr (SHARED) {
    float* const own = sm + w * STAGE;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        own[(db * 16 + v) * 64 + lane] = dk[db][v];
        own[((D / 32 + db) * 16 + v) * 64 + lane] = dv[db][v];
      }
    __syncthreads();
    for (int n = w; n < 2 * (D / 32); n += B32_WAVES) {
      const f32x16 sum = sum_records(sm, STAGE, n, lane);
      const bool is_v = n >= D / 32;
      if (krow < p.Sk) store(is_v ? dvp : dkp, is_v ? n - D / 32 : n, sum, is_v ? 1.f : p.scale);
    }
  } else if (krow < p.Sk) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      store(dkp, db, dk[db], p.scale);
      store(dvp, db, dv[db], 1.f);
    }
  }
}

// Query rows of the longest sequence (of a packed batch in shards Sq is what lies in one of them).
int64_t longest_rows(const BwdParams& p) { return (int64_t)p.Sq * (p.cu_q && p.map.P ? p.map.P : 1); }

// `rows` query rows, or keys, per workgroup.
template <auto kernel>
hipError_t launch(int smem, bool queries, int rows, BwdParams p, hipStream_t stream, int threads = BWD_THREADS) {
  const hipError_t e = spa_allow_dynamic_lds<kernel>(smem);
  if (e != hipSuccess) return e;
  dim3 grid;
  if (p.cu_q) {
    const int64_t longest = queries ? longest_rows(p) : (int64_t)p.Sk * (p.map.P ? p.map.P : 1);
    if (!spa_varlen_grid(p.H, p.B, queries ? p.lse_bh : p.total_k, longest, rows, 1, grid, p.numbered)) return hipErrorInvalidValue;
  } else {
    const int tiles = ((queries ? p.Sq : p.Sk) + rows - 1) / rows;
    if (tiles > 65535) return hipErrorInvalidValue;
    grid = spa_head_groups((int64_t)p.B * p.H, tiles);
  }
  hipLaunchKernelGGL(kernel, grid, dim3(threads), smem, stream, p);
  return hipGetLastError();
}

// What a launch of one of the forms below takes, in microseconds on a chip that does nothing else: its longest chain of tiles, or the work of all
// workgroups shared out over the CUs.  rows: what a workgroup owns (query rows of the dq kernel, keys of the dk / dv kernel), start: its
// start and end behind another's, alone: in a launch of few, tile: a tile of 64 of the other side (fitted to launches of 8 heads, 64 to 4096 causal rows,
// and of thousands of workgroups of 16 to 512 rows).
double launch_time(const BwdParams& p, bool queries, int rows, double start, double alone, double tile) {
  const int cus = spa_device_cus(), shards = p.cu_q && p.map.P ? p.map.P : 1;
  const double own = (double)(queries ? p.Sq : p.Sk) * shards;
  double other = (double)(queries ? p.Sk : p.Sq) * shards;  // rows of the other side
  if (p.causal && queries && own < other) other = own;
  const double chain = alone + tile * ceil(other / BWD_ROWS);
  // of a workgroup whose sequence has `o` rows on the other side
  const auto tiles = [&](double o) {
    const double n = (p.causal && (o + rows) / 2 < o ? (o + rows) / 2 : o) / BWD_ROWS;
    return n < 1 ? 1 : n;
  };
  double work;
  if (p.cu_q) {
    // The host knows the longest sequence and the mean of the others, and counts a batch of those: a workgroup for every sequence however short it is, and
    // one sequence that is longer than all others together as what it is (by the mean of all: one of 16384 rows and 100 of 128, 16 heads, 64 rows
    // and 64 keys instead of 256 and 128, dq 1450 -> 1560 us, dk / dv 1980 -> 2440).
    const double total = queries ? (double)p.lse_bh : (double)p.total_k, per_row = (queries ? (double)p.total_k : (double)p.lse_bh) / total;
    const double rest = p.B > 1 && total > own ? (total - own) / (p.B - 1) : 0;
    const bool alike = rest == own;
    const auto cost = [&](double s) {
      const double wgs = s <= rows ? 1 : alike ? ceil(s / rows) : s / rows + 0.5;
      return wgs * (start + tile * tiles(s * per_row));
    };
    work = p.H * (cost(own) + (p.B - 1) * cost(rest)) / cus;
  } else {
    // (Workgroups of one length go in whole rounds of one per CU; causal ones, the long ones first, and those of a ragged batch fill each other's gaps.
    // Not causal, training step, us, rounds as a fraction / whole: 12 heads of 1536 rows 126 / 93, 16 of 1280 97 / 82, 64 of 640 103 / 97, 32 of 1536 199 / 188.)
    const double rounds = (double)p.B * p.H * ceil(own / rows) / cus;
    work = (p.causal ? rounds : ceil(rounds)) * (start + tile * tiles(other));
  }
  return chain > work ? chain : work;
}

// D = 64: workgroups of 64 rows, or keys, up to which they are the faster ones.  Two run on a CU: all at once up to two a CU, and beyond that, causal, while
// the chains are long beside a workgroup's start and end (`rounds` - `start` / tiles, of workgroups of 128): the longest of the others decides, whose CU another
// one shares.  Both kernels, causal, us, with 128 rows and keys / 64 rows and 128 keys / 128 rows and 64 keys: 12 heads of 2811 rows 91.9 / 78.7 / 79.1; 8 of 4763 147.4 /
// 127.7 / 128.0; 16 of 2501 87.7 / 76.1 / 75.4; 4 x 16 of 674 33.6 / 35.1 / 38.2 (and with 64 of both 12 heads of 2811 72, 8 of 4763 116).  Of 1900 launches of 250 to 8000 rows, a quarter of them not causal, none got slower by it.
double most_64(const BwdParams& p, double rounds, double start) {
  const double of_128 = p.causal && !p.cu_q ? rounds - start / ((p.Sq + BWD_ROWS - 1) / BWD_ROWS) : 1.0;
  return 2.0 * spa_device_cus() * (of_128 > 1.0 ? of_128 : 1.0);
}

// The forms of the dq kernel, D = 128: 256 rows a workgroup (8 waves, two a SIMD, the K/V stream shared by twice the rows) where there are many;
// with fewer, 128 rows, or 64 (4 waves), whose waves share out the keys of a tile: more workgroups, each with a shorter chain.  Causal,
// us, 256 / 128 / 64 rows: 8 heads of 2048 rows 61.4 / 37.8 / 29.5, 4096 119 / 76.8 / 63.8, 8192 263 / 187 / 227; 16 of 4096 138 / 101 / 125; 32 of 512
// 20.5 / 15.4 / 12.6, 2048 76.4 / 58.5 / 79.2, 4096 181 / 196 / 259; 128 of 512 30.3 / 33.2 / 39.5.
// 128 rows on 4 waves that do not share, one a SIMD, where sequences are short (and for tensors of 2 GiB and more per (batch, head)): it starts the
// soonest.  Causal, us, 256 / 128 / 64 / 128 rows on 4 waves, 16 heads: 2000 sequences of 16 rows 988 / 1042 / 841 / 829, 1000 of 64 552 / 580 / 505 / 465, 500 of
// 128 376 / 381 / 514 / 367, 400 of 160 377 / 558 / 611 / 504, 200 of 320 424 / 491 / 587 / 460; 8 of 192 13.7 / 13.2 / 16.7 / 12.2, 8 of 128 10.8 / 10.4 / 9.2 / 10.4.
// D = 64: 128 rows, two workgroups to a CU, or 64 rows (most_64): 8 heads of 2048 rows 29.4 / 19.9, 4096 56.0 / 39.1, 8192
// 128 / 119; 16 of 2048 30.0 / 21.6; 32 of 1024 18.7 / 14.3, 2048 36.9 / 36.9; 128 of 512 16.8 / 19.4.
enum DqForm { DQ_128_PLAIN = 4, DQ_256 = 8, DQ_64 = 20, DQ_128 = 24 };  // the values of SPA_TUNE_BWD_DQ_WAVES
template <int D, int ADDR>
int dq_form(const BwdParams& p) {
  const int forced = spa_knob(SPA_KNOB_BWD_DQ_WAVES);
  if (D < 64 || ADDR == ADDR_BIG) return DQ_128_PLAIN;
  if (forced && (D == 128 || forced == DQ_64)) return forced;
  if (forced) return DQ_128_PLAIN;
  if (D == 64) {
    const double wgs = p.cu_q ? (double)p.H * ((double)p.lse_bh / 64 + p.B) : (double)p.B * p.H * ((p.Sq + 63) / 64);
    return wgs <= most_64(p, 2.25, 14.0) ? DQ_64 : DQ_128_PLAIN;
  }
  const double t256 = launch_time(p, true, 256, 6.0, 7.0, 1.76), t128 = launch_time(p, true, 128, 8.0, 8.4, 0.92);
  const double t64 = launch_time(p, true, 64, 7.5, 7.5, 0.69), plain = launch_time(p, true, 128, 5.5, 6.6, 1.2);
  const DqForm form = t64 < t128 ? (t64 < t256 ? DQ_64 : DQ_256) : t128 < t256 ? DQ_128 : DQ_256;
  return plain < (form == DQ_64 ? t64 : form == DQ_128 ? t128 : t256) ? DQ_128_PLAIN : form;
}

// Whether the dk / dv kernel takes 64 keys a workgroup.  Causal, us, 128 / 64 keys, D = 128: 8 heads of 512 rows 17.7 / 14.6, 2048 52.1 / 36.8, 4096
// 103 / 83.6, 8192 259 / 291; 16 of 2048 55.9 / 50.8, 4096 135 / 161; 32 of 512 19.5 / 17.0, 1024 33.9 / 35.5.  D = 64, two workgroups to a
// CU: 8 of 2048 35.1 / 24.3, 4096 67.9 / 51.2; 16 of 4096 86.5 / 86.1; 32 of 1024 22.2 / 18.5, 2048 47.0 / 48.9; not causal 8 of 2048 36.9 / 27.6, 16 of 2048 41.4 / 41.2.
template <int D, int ADDR>
bool keys_64(const BwdParams& p) {
  const int knob = spa_knob(SPA_KNOB_BWD_DKDV_FORM), form = knob > 3 ? knob - 2 : knob;  // (4, 5: the twins of 2, 3)
  if (D < 64 || ADDR == ADDR_BIG) return false;
  if (form > 1) return form == 2;
  if (D == 64) {
    const double wgs = p.cu_q ? (double)p.H * ((double)p.total_k / 64 + p.B) : (double)p.B * p.H * ((p.Sk + 63) / 64);
    return wgs <= (p.causal ? most_64(p, 2.1, 15.0) : 1.0 * spa_device_cus());
  }
  return launch_time(p, false, 64, 6.5, 6.5, 0.975) < launch_time(p, false, 128, 4.7, 4.7, 1.48);
}

template <typename T, int D, int ADDR = ADDR_PLAIN>
hipError_t launch_both(const BwdParams& p, hipStream_t stream) {
  hipError_t e = hipErrorInvalidValue;
  const int form = dq_form<D, ADDR>(p);
  if constexpr (D == 128 && ADDR != ADDR_BIG) {
    if (form == DQ_256) e = launch<flash_bwd_dq_kernel<T, D, 8, ADDR>>(DqCfg<D, 8>::SMEM, true, 256, p, stream, 512);
    if (form == DQ_128) e = launch<flash_bwd_dq_kernel<T, D, 8, ADDR, 2>>(DqCfg<D, 8, 2>::SMEM, true, 128, p, stream, 512);
  }
  if constexpr (D >= 64 && ADDR != ADDR_BIG)
    if (form == DQ_64) e = launch<flash_bwd_dq_kernel<T, D, 4, ADDR, 2>>(DqCfg<D, 4, 2>::SMEM, true, 64, p, stream);
  if (form == DQ_128_PLAIN) e = launch<flash_bwd_dq_kernel<T, D, 4, ADDR>>(DqCfg<D, 4>::SMEM, true, 128, p, stream);
  if (e != hipSuccess) return e;
  const bool narrow = keys_64<D, ADDR>(p);
  if constexpr (D == 128 && ADDR == ADDR_PLAIN)
    if (const int form = spa_knob(SPA_KNOB_BWD_DKDV_FORM); form == 1 || form > 3)
      return narrow ? launch<flash_bwd_dkdv_kernel<T, D, false, ADDR, 2>>(DkvCfg<D>::SMEM, false, 64, p, stream)
                    : launch<flash_bwd_dkdv_kernel<T, D, false>>(DkvCfg<D>::SMEM, false, 128, p, stream);
  if constexpr (D >= 64 && ADDR != ADDR_BIG)
    if (narrow) return launch<flash_bwd_dkdv_kernel<T, D, true, ADDR, 2>>(DkvCfg<D>::SMEM, false, 64, p, stream);
  return launch<flash_bwd_dkdv_kernel<T, D, true, ADDR>>(DkvCfg<D>::SMEM, false, 128, p, stream);
}

template <typename T, int D>
hipError_t launch_other(const BwdParams& p, hipStream_t stream) {
  if (!p.map.P) return launch_both<T, D, ADDR_BIG>(p, stream);
  if (p.big || !p.grads_in_t) return hipErrorInvalidValue;
  return launch_both<T, D, ADDR_MAP>(p, stream);
}

}  // namespace

// This file makes two objects: compiled with SPA_BWD_OTHER_UNIT it holds the re-based variants of the 16-bit kernels and
// those for rows in shards and nothing else, without it everything else (so that the two parts compile side by side).
#ifdef SPA_BWD_OTHER_UNIT
hipError_t spa_launch_bwd16_other(const BwdParams& p, int D, int dtype, hipStream_t stream) {
  if (dtype == 1) {
    if (D == 128) return launch_other<__bf16, 128>(p, stream);
    if (D == 64) return launch_other<__bf16, 64>(p, stream);
    if (D == 32) return launch_other<__bf16, 32>(p, stream);
  } else if (dtype == 2) {
    if (D == 128) return launch_other<_Float16, 128>(p, stream);
    if (D == 64) return launch_other<_Float16, 64>(p, stream);
    if (D == 32) return launch_other<_Float16, 32>(p, stream);
  }
  return hipErrorInvalidValue;
}
#else
hipError_t spa_launch_bwd16_other(const BwdParams& p, int D, int dtype, hipStream_t stream);

// fp32: whether the waves of a workgroup share out the tiles (SHARED).  A launch lasts as long as its longest chain of tiles or as the
// work of all SIMDs, whichever is more; sharing quarters the chain, and costs the workgroup's sums and, where all SIMDs are busy, 6 to 16 %
// ([1, 2048, 32, 128] causal 1178 us, shared 1366).  Of 14 launches of 128 to 2048 rows the rule takes the faster form in each.
bool tiles_shared(const BwdParams& p) {
  const int knob = spa_knob(SPA_KNOB_FWD32_SPLIT);
  if (p.Sq > 65535 * B32_ROWS || p.Sk > 65535 * B32_ROWS) return false;
  if (knob) return knob == 2;
  const double rows = (p.Sq + 31) / 32, keys = (p.Sk + 31) / 32;
  const double all = p.cu_q ? (double)p.H * (p.lse_bh / 32 + p.B) : (double)p.B * p.H * rows;  // row tiles of the launch
  const double chain = p.causal && rows < keys ? rows : keys, work = all * (p.causal ? chain / 2 : chain) / (4 * spa_device_cus());
  const double shared = chain / B32_WAVES > 1.2 * work ? chain / B32_WAVES : 1.2 * work;
  return shared + 0.5 < (chain > work ? chain : work);
}
template <int D>
hipError_t launch32(const BwdParams& p, hipStream_t stream) {
  typedef Bwd32Cfg<D> C;
  if (tiles_shared(p)) {
    const hipError_t e = launch<flash_bwd32_dq_kernel<D, true>>(C::SMEM_SHARED, true, 32, p, stream);
    return e != hipSuccess ? e : launch<flash_bwd32_dkdv_kernel<D, true>>(C::SMEM_SHARED, false, 32, p, stream);
  }
  const hipError_t e = launch<flash_bwd32_dq_kernel<D, false>>(C::SMEM_DQ, true, 128, p, stream);
  return e != hipSuccess ? e : launch<flash_bwd32_dkdv_kernel<D, false>>(C::SMEM_DKV, false, 128, p, stream);
}

// Returns hipSuccess, or hipErrorInvalidValue for an unsupported (dtype, D).
hipError_t spa_launch_flash_bwd(BwdParams p, int D, int dtype, hipStream_t stream) {
  if ((p.big || p.map.P) && dtype != 0) return spa_launch_bwd16_other(p, D, dtype, stream);
  if (dtype == 1) {
    if (D == 128) return launch_both<__bf16, 128>(p, stream);
    if (D == 64) return launch_both<__bf16, 64>(p, stream);
    if (D == 32) return launch_both<__bf16, 32>(p, stream);
  } else if (dtype == 2) {
    if (D == 128) return launch_both<_Float16, 128>(p, stream);
    if (D == 64) return launch_both<_Float16, 64>(p, stream);
    if (D == 32) return launch_both<_Float16, 32>(p, stream);
  } else if (dtype == 0) {
    if (D == 128) return launch32<128>(p, stream);
    if (D == 64) return launch32<64>(p, stream);
    if (D == 32) return launch32<32>(p, stream);
  }
  return hipErrorInvalidValue;
}
#endif  // SPA_BWD_OTHER_UNIT
