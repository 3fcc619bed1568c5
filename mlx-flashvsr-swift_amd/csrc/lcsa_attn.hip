// Block-sparse flash attention over 128x128 blocks for gfx950 (MI355X).
//
// Reference semantics: the Metal kernel of SparseAttention.swift:17-154 (launched at :180-185) and the dense path
// blockMaskedAttention (DiT.swift:279-313): per head, o = softmax(q k^T / sqrt(128)) v over the listed key blocks,
// fp32 online softmax, a query block with no listed key block writes zeros.
//
// bf16 (the production lane): a persistent walk over rows (head, 128-query block); a workgroup = 4 wave64s x 32
// queries, two waves per SIMD; K/V tiles of 32 keys reach LDS by direct buffer->LDS copies into 4-slot rings;
// S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_32x32x16_bf16 so each lane owns one query row; the softmax keeps a fixed
// reference per row (see the kernel's comment). fp32 (the parity lane): 4 wave64s x 32 queries, every fp32 operand
// split into three bf16 parts and multiplied on the bf16 matrix cores, with a lazy online-softmax rescale. In
// both, calls with few rows split the rows' key lists into pieces that a second kernel merges.
#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "common.hpp"

namespace fvsr {

__device__ __forceinline__ float pair_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) char lds_char;


// O^T += A B on the matrix core. The library is compiled with the MFMA VGPR form (-amdgpu-mfma-vgpr-form): the score
// MFMAs, whose results the VALU reads, and this accumulation write VGPRs (the working set, about 230 registers, fits
// the 256 of two waves per SIMD). The accumulation is the compiler's builtin, so it sees every hazard and keeps one
// register assignment for O across the walk's control paths (the reference raise); successive accumulations into
// one block are >= 7 MFMAs apart.
__device__ __forceinline__ void mfma_acc(f32x16& acc, const bf16x8& a, const bf16x8& b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}
// >= 19 wait states after the last MFMA of a walk (the compiler also inserts what it needs)
__device__ __forceinline__ void acc_drain() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory"); }

// Lazy online-softmax rescale. The running reference max m_run (log2 domain, per query row) is raised only when a
// tile's row max exceeds it by more than 8, i.e. a factor 2^8: exponentials then stay <= 256 (no overflow in fp32 or
// bf16) and the softmax is mathematically unchanged, while the O/l rescale — a multiply over the whole accumulator —
// runs only on the few tiles where some row of the wave grows (wave-uniform branch). Returns the max to subtract.
template <int NACC>
__device__ __forceinline__ float rescale_if_grown(float mxc, float& m_run, float& l_run, f32x16 (&acc)[NACC]) {
  const bool grow = mxc > m_run + 8.f;
  if (__ballot(grow) != 0) {
    const float m_new = grow ? mxc : m_run;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);   // m_run = -inf -> 0; unchanged row -> 1
    l_run *= alpha;
#pragma unroll
    for (int d = 0; d < NACC; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[d][r] *= alpha;
    m_run = m_new;
  }
  return m_run == -INFINITY ? 0.f : m_run;
}

// ------------------------------------------------------------------------------------------------------------
// bf16
// ------------------------------------------------------------------------------------------------------------
// One workgroup = one (head, 128-query block) at a time, two workgroups per CU. QG = 1 (the default): 4 wave64s x 32
// queries, two waves per SIMD (at most 256 registers each), so one wave's LDS, memory and VALU stalls are covered by
// the other's MFMAs. QG = 2: 2 wave64s x 64 queries held as two 32-query groups, one wave per SIMD; every K or V
// operand read from LDS then feeds two MFMAs.
//
// Keys stream in tiles of 32 (a quarter of a 128-key block). K and V tiles land in two LDS rings of kSlots slots by
// buffer_load ... lds (16 B per lane, no VGPR staging); a tile's rows are 256 B (one head) with the 16-byte chunks
// XOR-swizzled by row so the ds_read_b128 (K) and ds_read_b64_tr_b16 (V^T) operand reads are bank-conflict free.
// While tile T is processed (step T), K of tile T+4 and V of tile T+2 are requested; each step ends by waiting for
// the copies of the step before it, so a tile is in LDS a step before the step that first reads it.
//
// Softmax with a lazily raised reference per query row: S = K Q^T in fp32 from the bf16 inputs (keys that do not
// take part score -2^100, by a select on the rare tile with fewer than 32 keys: a ragged end, an index outside
// [0, nk), the tile past the walk's end), then
// P = exp2(c S - m) with one v_fma per score (c = log2(e)/sqrt(128), applied to the fp32 scores as the reference
// does, SparseAttention.swift:96; m, the row's reference, first the exact max of its first tile). A tile whose
// partial row sum exceeds 2^32 (its scores outgrew the reference by about 27 or more, in log2 units) raises the
// reference to the tile's max: its exponentials are recomputed and O and l rescaled (a wave-uniform branch, rare:
// rows with sharp attention raise it a few times). Rows whose exponentials all underflowed (a reference from a tile
// with no valid key, and every real score 2^-32 below it) make the workgroup redo its rows exactly (row-max pass,
// then attention with that max). The result is the softmax whatever the reference is.
//
// Software pipeline per wave, step T: the exponentials of S(T) are issued between the MFMAs of PV(T-1) and QK(T+1),
// so the VALU work hides under matrix-core time. The walk is unrolled by one 128-key block (4 steps); block indices
// are read three blocks ahead so no scalar load latency sits on the step.
namespace {

constexpr int kTileKeys = 32;
constexpr int kRowBytes = kHeadDim * 2;                // one head of one token, bf16
constexpr int kTileBytes = kTileKeys * kRowBytes;      // 8 KB
constexpr int kSlots = 4;                              // per ring: slot of tile T = T mod 4 = its quarter of the block
constexpr int kVRing = kSlots * kTileBytes;            // byte offset of the V ring
constexpr float kMaskedScore = -1.2676506e30f;         // -2^100: exp2 of a masked key is exactly 0
constexpr float kGrowSum = 4294967296.f;               // 2^32: a larger partial row sum raises the reference
constexpr int kMaxPersistentWgs = 1024;                // persistent grid cap (the order kernel's first-row deal)

// 16-byte chunk swizzles. K: the 8 (or 16) lanes one ds_read_b128 cycle serves read 8 (16) consecutive rows of one
// chunk -> distinct positions. V: a ds_read_b64_tr_b16 half-wave (32 lanes, 256 B, one pass over the 64 banks of a
// 256-byte row) reads 4 consecutive rows (a multiple of 4 apart) x 4 adjacent chunks (two 16-lane groups of 2):
// XOR-ing the chunk index with 4 * (row mod 4) puts the 4 rows' aligned 4-chunk groups on 4 different groups, so the
// 32 lanes cover all 64 banks once (the SQ_LDS_BANK_CONFLICT counter reads 0; the former (2 * row) mod 16 swizzle
// left every second cycle a conflict).
__device__ __forceinline__ int swz_k(int r) { return r & 15; }
__device__ __forceinline__ int swz_v(int r) { return (r & 3) << 2; }

// s_waitcnt vmcnt(n) lgkmcnt(0) (gfx9 encoding: vmcnt bits [3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8])
#define FVSR_WAIT_VM_LGKM0(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | ((((n) >> 4) & 3) << 14) | (7 << 4))

// 16 bytes per lane from a buffer straight into LDS at lds_base + OFF + 16 * lane. Issued as inline assembly so the
// compiler does not order every later LDS read behind it: the kernel orders the copies itself (vmcnt + barrier).
// M0 is written without a clobber declaration (the compiler reserves it); nothing else in these kernels uses M0. It
// is loaded with s_mov_b32 from an address computed outside the asm. GFX9 requires one wait state between an SALU
// write of M0 and an LDS DMA that reads it; the compiler inserts it for its own code but not inside an asm
// statement, so the s_nop is written out.
// The row's offset `voff` and the block's offset `boff` are added into the one VGPR offset (the SGPR offset is 0):
// the raw buffer's range check covers the VGPR offset and the instruction offset, not the SGPR offset, so only an
// offset held there makes a row past the buffer (a ragged last block, a listed index outside [0, nk), the tiles past
// the end of the walk, whose block offset is the buffer's size) load zeros without touching memory.
template <int OFF>
__device__ __forceinline__ void dma16(u32x4 rsrc, uint32_t lds_base, int voff, int boff) {
  const uint32_t off = (uint32_t)voff + (uint32_t)boff;   // voff holds the head's offset, inside the buffer: < 2^32
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds_base + OFF),
               "v"(off), "s"(rsrc));
}

__device__ __forceinline__ u32x4 buffer_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)base;
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}


}  // namespace

// The next position of the per-XCD queues of attn_order_kernel's dealt order, starting with this workgroup's XCD
// (dispatch is round-robin over the XCDs: XCD of workgroup b = b % 8), then stealing from the others; `rows` when
// every queue is empty. Queue y holds, wave by wave, the positions w * grid + y + 8 i, i < per_y = ceil((grid - y)
// / 8); its counter (counters[8 y]) starts past the first wave, which the workgroups take without it. Positions
// grow with the counter, so the first one past `rows` means the queue is empty. Called by one thread.
__device__ __forceinline__ int next_dealt_item(int32_t* counters, int rows) {
  const int grid = (int)gridDim.x;
  for (int t = 0; t < kXcds; ++t) {
    const int y = ((int)blockIdx.x + t) & (kXcds - 1);
    const int per = (grid - y + kXcds - 1) / kXcds;
    if (per <= 0) continue;
    const int k = atomicAdd(counters + 8 * y, 1);
    const int p = (k / per) * grid + y + kXcds * (k % per);
    if (p < rows) return p;
  }
  return rows;
}

constexpr int kMaxSplitItems = 512;   // the partial results of a call: at most 34 MB
constexpr int kMaxSplitRows = 256;    // rows whose lists are split: a row or two a thread in split_item
constexpr int kMaxPieces = 32;        // the merge walks a row's pieces one after another

// An item: a row (head-major, 128 queries), or one of the `pieces` pieces of a row's key list: entries [b0, b0 + nblocks).
struct AttnItem {
  int row, h, qb, b0, nblocks;
  int slot, pieces;   // pieces > 1: the item's partial result
};

// Splits the rows' key lists into at most G pieces of about the same length: T, the most blocks of a piece, is the smallest
// of 64 candidates from max(min_blocks, longest / kMaxPieces, blocks / G) up to the longest list with sum max(1, ceil(len / T)) <= G
// (2 rows <= G, so the last always fits), and a row of n = ceil(len / T) pieces is cut at len p / n. The pieces number the
// rows in order. Where the longest list is at most split_slow / 16 T + split_cost blocks, pieces do not pay and every row is
// one. Every workgroup finds the same T and then its own piece; a row's first piece leaves (n << 16 | number) in
// plan[row] for the merge. `sm` is LDS for kMaxSplitRows + 4 x 64 + 8 ints. Called by the whole workgroup of THREADS; false for a
// workgroup without an item. Costs about a microsecond: one round trip for the lengths and four barriers.
template <int THREADS>
__device__ __forceinline__ bool split_item(const AttnArgs& a, const int32_t* __restrict__ kcnt, int rows, int32_t* plan,
                                           int* sm, AttnItem& it) {
  constexpr int kWaves = THREADS / 64, kPer = kMaxSplitRows / THREADS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int* const lens = sm;                          // [kMaxSplitRows]
  int* const cand = sm + kMaxSplitRows;          // [kWaves][64]
  int* const tot = cand + kWaves * 64;           // [2 kWaves]
  // thread tid holds rows kPer tid .. kPer tid + kPer - 1 (length 0 past the last row)
  int len[kPer], sum = 0, mx = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int r = kPer * tid + i;
    len[i] = r < rows ? max(0, min(kcnt[r], a.nk_stride)) : 0;
    lens[r] = len[i];
    sum += len[i];
    mx = max(mx, len[i]);
  }
  sum = wave_scan_dpp(sum);
  for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o));
  if (lane == 63) {
    tot[wave] = sum;
    tot[kWaves + wave] = mx;
  }
  __syncthreads();
  sum = mx = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    sum += tot[w];
    mx = max(mx, tot[kWaves + w]);
  }
  const int G = a.split_items;
  const int t0 = max(max(a.split_min, (mx + kMaxPieces - 1) / kMaxPieces), (sum + G - 1) / G);
  const int dt = max(1, (mx - t0 + 62) / 63);   // t0 + 63 dt >= mx
  // ceil(len / T) in fp32: floor((len + T - 1/2) / T), at least 1 / (2 T) from an integer, so exact up to lists of a million
  // entries; beyond, a count may be one too many, alike in every workgroup, which the cuts do not mind (the last candidate
  // still fits: G >= 2 rows)
  auto pieces_of = [](int len, float t, float inv) -> int { return max(1, (int)((len + t - 0.5f) * inv)); };
  const float tc = (float)(t0 + lane * dt), ic = 1.f / tc;
  // lane l tries T = t0 + l dt; each wave counts the pieces of its own rows
  int n = 0;
  const int r_end = min(rows, (wave + 1) * kPer * 64);
  for (int r = wave * kPer * 64; r < r_end; r += 8) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const i32x4 x = *(const i32x4*)(lens + r), y = *(const i32x4*)(lens + r + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      n += r + e < r_end ? pieces_of(x[e], tc, ic) : 0;
      n += r + 4 + e < r_end ? pieces_of(y[e], tc, ic) : 0;
    }
  }
  cand[wave * 64 + lane] = n;
  __syncthreads();
  n = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) n += cand[w * 64 + lane];
  const int best = __ffsll((unsigned long long)__ballot(n <= G)) - 1;   // lane 63 fits
  const int Tb = t0 + best * dt;
  const bool whole = 16ll * mx <= (int64_t)a.split_slow * Tb + 16 * a.split_cost;
  const int items = whole ? rows : __builtin_amdgcn_readlane(n, best);
  const float T = (float)Tb, iT = 1.f / T;
  // XCD x (workgroups b with b % 8 = x) takes a contiguous range of the pieces, whose key blocks overlap
  const int xcd = blockIdx.x % kXcds, idx = blockIdx.x / kXcds;
  const int q = items / kXcds, rem = items % kXcds;
  const int mine = idx < q + (xcd < rem ? 1 : 0) ? xcd * q + min(xcd, rem) + idx : -1;
  // the row that holds piece `mine`
  int c[kPer], csum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    c[i] = kPer * tid + i < rows ? (whole ? 1 : pieces_of(len[i], T, iT)) : 0;
    csum += c[i];
  }
  int at = wave_scan_dpp(csum) - csum;
  // pieces of the waves before: their rows, or their candidates' counts
  for (int w = 0; w < wave; ++w) at += whole ? kPer * 64 : __builtin_amdgcn_readfirstlane(cand[w * 64 + best]);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    if (mine >= at && mine < at + c[i]) {
      tot[0] = kPer * tid + i;
      tot[1] = mine - at;
      tot[2] = c[i];
    }
    at += c[i];
  }
  __syncthreads();
  if (mine < 0) return false;
  const int row = __builtin_amdgcn_readfirstlane(tot[0]), piece = __builtin_amdgcn_readfirstlane(tot[1]);
  it.pieces = __builtin_amdgcn_readfirstlane(tot[2]);
  const int n_row = __builtin_amdgcn_readfirstlane(lens[row]);
  it.slot = mine;
  it.row = row;
  it.h = row / a.nq;
  it.qb = row - it.h * a.nq;
  it.b0 = (int)((int64_t)n_row * piece / it.pieces);
  it.nblocks = (int)((int64_t)n_row * (piece + 1) / it.pieces) - it.b0;
  if (piece == 0 && tid == 0) plan[row] = it.pieces << 16 | mine;
  __syncthreads();   // the LDS is free
  return true;
}

// the pieces of a row that lists n blocks, where rows are cut in a.pieces equal ones: a single block stays whole
__device__ __forceinline__ int row_pieces(const AttnArgs& a, int n) { return n <= 1 ? 1 : a.pieces; }

// The next item of this workgroup. DIRECT (every item has a workgroup of its own): one item, a piece of the split or the
// XCD-remapped workgroup index as piece (index / rows of a.pieces) of row (index % rows). Else the row at its position of the order's first wave, then of its XCD's
// queue. Called by the whole workgroup; false when nothing is left.
template <bool DIRECT, int THREADS>
__device__ __forceinline__ bool next_item(const AttnArgs& a, const int32_t* __restrict__ kcnt,
                                          int32_t* __restrict__ order, int32_t* __restrict__ counter, int rows,
                                          bool first, int tid, int* item_s, int* sm, AttnItem& it) {
  if constexpr (DIRECT) {
    if (a.split_items > 0) return split_item<THREADS>(a, kcnt, rows, order, sm, it);
    it.slot = xcd_remap(blockIdx.x, gridDim.x);   // neighbouring items: neighbouring rows' same pieces
    const int piece = it.slot / rows;
    it.row = it.slot - piece * rows;
    it.h = it.row / a.nq;
    it.qb = it.row - it.h * a.nq;
    const int n = max(0, min(kcnt[it.row], a.nk_stride));
    it.pieces = row_pieces(a, n);
    it.b0 = (int)((int64_t)n * piece / it.pieces);
    it.nblocks = (int)((int64_t)n * (piece + 1) / it.pieces) - it.b0;
    return piece < it.pieces;
  } else {
    int p = blockIdx.x;
    if (!first) {
      if (tid == 0) *item_s = next_dealt_item(counter, rows);
      __syncthreads();
      p = *item_s;
      __syncthreads();
    }
    if (p >= rows) return false;
    it.row = order[p];
  }
  it.h = it.row / a.nq;
  it.qb = it.row - it.h * a.nq;
  it.b0 = 0;
  it.nblocks = max(0, min(kcnt[it.row], a.nk_stride));
  it.pieces = 1;
  return true;
}

// An item that lists no block: a whole row is zeros (SparseAttention.swift:47-53; DiT.swift:300-304), a piece is a partial
// result of weight 0.
template <typename T>
__device__ __forceinline__ void attn_empty_item(const AttnArgs& a, const AttnItem& it, T* __restrict__ O, int tid,
                                                int threads) {
  constexpr int VN = 16 / sizeof(T), kVecs = kHeadDim / VN;
  if (it.pieces > 1) {
    for (int e = tid; e < kBlock; e += threads) a.part_ml[(int64_t)it.slot * 2 * kBlock + kBlock + e] = 0.f;
    return;
  }
  for (int e = tid; e < kBlock * kVecs; e += threads) {
    const int64_t row = (int64_t)it.qb * kBlock + e / kVecs;
    if (row < a.lq) *(u32x4*)(O + a.out_row(row) * a.ld + it.h * kHeadDim + (e % kVecs) * VN) = u32x4{0, 0, 0, 0};
  }
}

// The result of 32 queries (group `group` of the item's four; lane l holds query l % 32, dims 32 dt + 8 r4 + 4 (l / 32) + e
// at acc[dt][4 r4 + e]) from the unnormalised accumulator, the softmax sum l and the reference m (log2 units): the output
// row, or the piece's partial result in register order (1 KB per store instruction).
template <bool DIRECT, typename T>
__device__ __forceinline__ void attn_store(const AttnArgs& a, const AttnItem& it, int group,
                                           const f32x16 (&acc)[4], float m, float l, T* __restrict__ O) {
  typedef T Tx4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, g = lane >> 5, l32 = lane & 31;
  if (DIRECT && it.pieces > 1) {
    float* const po = a.part_o + ((int64_t)it.slot * 4 + group) * (32 * kHeadDim) + 4 * lane;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[i >> 2][4 * (i & 3) + e];
      *(f32x4*)(po + i * 256) = v;
    }
    if (g == 0) {
      float* const ml = a.part_ml + (int64_t)it.slot * 2 * kBlock + group * 32 + l32;
      ml[0] = m;
      ml[kBlock] = l;
    }
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int64_t qrow = (int64_t)it.qb * kBlock + group * 32 + l32;
  if (qrow >= a.lq) return;
  T* const orow = O + a.out_row(qrow) * a.ld + it.h * kHeadDim;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    Tx4 ov;
#pragma unroll
    for (int e = 0; e < 4; ++e) ov[e] = (T)(acc[i >> 2][4 * (i & 3) + e] * inv);
    *(Tx4*)(orow + 8 * i + 4 * g) = ov;
  }
}

// LDS operand requests of chunk / pair j >= 2 (j = 0, 1: micro-round 0), in micro-rounds of a step with QG query
// groups per wave: 7 (QG 2) or 4 (QG 1) micro-rounds before the QK MFMA that uses them, micro-round 0 at the earliest
template <int QG>
constexpr int attn_read_at(int j) {
  const int r = 2 * QG * j - (QG == 2 ? 7 : 4);
  return r > 0 ? r : 0;
}

template <int QG, bool DIRECT>
__global__ __attribute__((amdgpu_flat_work_group_size(256 / QG, 256 / QG), amdgpu_waves_per_eu(3 - QG, 3 - QG)))
void attn_bf16_kernel(AttnArgs a, const int32_t* __restrict__ kidx, const int32_t* __restrict__ kcnt,
                      const bf16* __restrict__ Q, bf16* __restrict__ O,
                      int32_t* __restrict__ order, int32_t* __restrict__ counter) {
  __shared__ __attribute__((aligned(1024))) char smem[2 * kVRing];
  __shared__ int item_s;

  // QG 32-query groups per wave: 4 / QG waves of 32 * QG queries; every wave copies 8 * QG rows of each tile
  constexpr int kWaves = 4 / QG, kThreads = 64 * kWaves, kQW = 32 * QG, kWaveRows = 8 * QG;
  constexpr int kDmaK = 2 * QG, kDmaStep = 4 * QG;   // per wave: copies of one K (V) tile, of one step
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  const int rows = a.heads * a.nq;
  // With more rows than resident workgroups the walk is persistent. attn_order_kernel sorts the rows longest key list
  // first and deals every wave of gridDim.x of them by XCD (re-sorted by row id, XCD x holds positions x, x + 8, ..
  // of the wave: one contiguous row range, whose key lists overlap). Workgroup b starts on position b of the first
  // wave; after that it takes the next position of its XCD's queue (positions x, x + 8, .. of the first wave, then
  // of the second, ...) and, once that queue is empty, of the other XCDs' queues in turn. So the long rows start
  // early, the rows running together on one XCD share key blocks in its L2, and the short ones balance the tail.
  for (bool first = true;; first = false) {
  AttnItem it;
  if (!next_item<DIRECT, kThreads>(a, kcnt, order, counter, rows, first, tid, &item_s, (int*)smem, it)) break;
  if (it.nblocks <= 0) {
    attn_empty_item<bf16>(a, it, O, tid, kThreads);
    if constexpr (DIRECT) break;
    else continue;
  }
  const int h = it.h, qb = it.qb, nblocks = it.nblocks;
  const int hc = h * kHeadDim;
  const int32_t* __restrict__ klist = kidx + (int64_t)it.row * a.nk_stride + it.b0;

  // Q as the B operand of S^T = K Q^T (the bf16 inputs as they are; the scale c is applied to the fp32 scores):
  // group q holds queries qb*128 + kQW*wave + 32*q + l32, lane (query, k-half g) dims 16t + 8g .. +7
  bf16x8 qop[QG][8];
#pragma unroll
  for (int q = 0; q < QG; ++q) {
    const int64_t qrow = (int64_t)qb * kBlock + wave * kQW + q * 32 + l32;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      bf16x8 x = bf16x8{};
      if (qrow < a.lq) x = *(const bf16x8*)(Q + qrow * a.ld + hc + 16 * t + 8 * g);
      qop[q][t] = x;
    }
  }

  // tile loads: the buffer spans the physical K/V rows; a row past it reads as 0, so a ragged last block, a listed
  // index outside [0, nk) and the tiles past the end of the walk load zeros without per-lane guards. K/V rows are
  // token-major (head h's 128 channels at 256 h bytes of each row) or head-major (a KV ring: head h's rows from
  // h * kv_head_stride on, 256 bytes each; every block whole, so no row past a head's region is read)
  const uint32_t row_bytes = (uint32_t)a.kv_ld * 2;
  const uint32_t range = (uint32_t)a.kv_bytes;
  const int head_off = (int)(h * a.kv_head_stride * 2);
  const u32x4 krs = buffer_rsrc(a.k, range), vrs = buffer_rsrc(a.v, range);
  // a DMA load writes 1 KB of LDS (lane i -> bytes 16i..16i+15) = 4 rows; wave w fills rows kWaveRows * w ..
  int voff_k[kDmaK], voff_v[kDmaK];
#pragma unroll
  for (int p = 0; p < kDmaK; ++p) {
    const int r = wave * kWaveRows + 4 * p + (lane >> 4), pos = lane & 15;
    voff_k[p] = r * (int)row_bytes + head_off + ((pos ^ swz_k(r)) << 4);
    voff_v[p] = r * (int)row_bytes + head_off + ((pos ^ swz_v(r)) << 4);
  }
  const uint32_t smem_lds = lds_addr(smem);
  const uint32_t dma_base = smem_lds + wave * kWaveRows * kRowBytes;
  // buffer byte offset of block j's first row (j outside [0, nk): past the buffer -> zeros)
  auto block_soff = [&](int j) -> int {
    return (unsigned)j < (unsigned)a.nk ? (int)(a.map.row(j) * row_bytes) : (int)range;
  };
  const int sub_bytes = kTileKeys * (int)row_bytes;   // 32 rows
  // K / V of quarter SUB of the block at soff into ring slot SLOT
  auto issue_k = [&](auto slot_c, int soff) {
    constexpr int SLOT = decltype(slot_c)::value;
    static_for<0, kDmaK>([&](auto p_c) {
      constexpr int P = decltype(p_c)::value;
      dma16<SLOT * kTileBytes + P * 4 * kRowBytes>(krs, dma_base, voff_k[P], soff);
    });
  };
  auto issue_v = [&](auto slot_c, int soff) {
    constexpr int SLOT = decltype(slot_c)::value;
    static_for<0, kDmaK>([&](auto p_c) {
      constexpr int P = decltype(p_c)::value;
      dma16<kVRing + SLOT * kTileBytes + P * 4 * kRowBytes>(vrs, dma_base, voff_v[P], soff);
    });
  };
  // one of the kDmaK copies (rows 4P .. 4P+3 of this wave's share) of K / V into ring slot SLOT
  auto dma_k = [&](auto slot_c, auto p_c, int soff) {
    constexpr int SLOT = decltype(slot_c)::value, P = decltype(p_c)::value;
    dma16<SLOT * kTileBytes + P * 4 * kRowBytes>(krs, dma_base, voff_k[P], soff);
  };
  auto dma_v = [&](auto slot_c, auto p_c, int soff) {
    constexpr int SLOT = decltype(slot_c)::value, P = decltype(p_c)::value;
    dma16<kVRing + SLOT * kTileBytes + P * 4 * kRowBytes>(vrs, dma_base, voff_v[P], soff);
  };
  // walked block b: buffer offset of its first row (past the buffer past the end of the walk) and its keys taking
  // part (0 outside [0, nk); else up to 128, fewer for a ragged last block). A walked block's entry is its key block
  // index, -1 past the end. The loop loads each entry one block before it derives the offset and key count from it,
  // so the load's wait is covered by the waits of the steps in between.
  auto walk_entry = [&](int b) -> int { return b < nblocks ? klist[b] : -1; };
  auto entry_soff = [&](int b, int j) -> int { return b < nblocks ? block_soff(j) : (int)range; };
  auto entry_keys = [&](int b, int j) -> int {
    if (b >= nblocks || (unsigned)j >= (unsigned)a.nk) return 0;
    return (int)min<int64_t>(kBlock, a.lk - (int64_t)j * kBlock);
  };
  auto walk_soff = [&](int b) -> int { return entry_soff(b, walk_entry(b)); };
  auto walk_keys = [&](int b) -> int { return entry_keys(b, walk_entry(b)); };
  auto sub_valid = [&](int keys, int sub) -> int { return min(max(keys - sub * kTileKeys, 0), kTileKeys); };

  // LDS operand addresses within a slot. K: row l32, chunk 2t+g. V^T (ds_read_b64_tr_b16): 16-lane group G, member
  // mm reads row 16u + 8ab + 4(G/2) + mm/4, bf16 columns 32dt + 16(G%2) + 4(mm%4) .. +3.
  int k_off[8], v_off[4];
#pragma unroll
  for (int t = 0; t < 8; ++t) k_off[t] = l32 * kRowBytes + (((2 * t + g) ^ swz_k(l32)) << 4);
  const int G = lane >> 4, mm = lane & 15;
  const int vr = 4 * (G >> 1) + (mm >> 2);   // + 16u + 8ab: the swizzle depends on the row mod 4 only
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
    v_off[dt] = vr * kRowBytes + (((4 * dt + 2 * (G & 1) + ((mm & 3) >> 1)) ^ swz_v(vr)) << 4) + (mm & 1) * 8;

  f32x16 acc[QG][4];
  float l_run[QG], m_row[QG], part_max[QG], m_ref[QG], negm[QG];
  constexpr float kNoKey = -1e29f;   // a raw row max below this saw masked keys only
  const float c_scale = a.c;         // softmax scale * log2(e)
  // the reference (log2 units, fp32) of each query row: P = exp2(c S - m), one v_fma per score
  auto set_ref = [&](int q, float m) {
    m_ref[q] = m;
    negm[q] = -m;
  };
  // the reference of a raw row max (masked keys only: 0)
  auto ref_of = [&](float mx) -> float { return mx > kNoKey ? mx * c_scale : 0.f; };
  // The walk lists selected blocks only, so its tiles are whole (32 keys) but for a ragged last block, a listed
  // index outside [0, nk) and the tile past the end of the walk, whose rows all load as zeros. S starts at zero and,
  // on a tile with fewer than 32 keys taking part (a wave-uniform branch), the scores of the keys at or past `valid`
  // are set to -2^100 afterwards: their exponentials are exactly 0.
  // Lane element i of a 32 x 32 MFMA result is key row 8 (i / 4) + 4 g + i % 4.
  auto mask_tile = [&](f32x16& s, int valid) {
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 8 * (i >> 2) + 4 * g + (i & 3) >= valid ? kMaskedScore : s[i];
  };
  lds_char* const lds = (lds_char*)(uintptr_t)smem_lds;
  // S^T = K Q^T (keys that do not take part: -2^100) for every group, K from ring slot SLOT
  auto qk = [&](auto slot_c, int valid, f32x16 (&s)[QG]) {
    constexpr int SLOT = decltype(slot_c)::value;
    bf16x8 kk[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) kk[t] = *(const lds_bf16x8*)(lds + SLOT * kTileBytes + k_off[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int q = 0; q < QG; ++q)
        s[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kk[t], qop[q][t], t > 0 ? s[q] : f32x16{}, 0, 0, 0);
    if (valid < kTileKeys) {
#pragma unroll
      for (int q = 0; q < QG; ++q) mask_tile(s[q], valid);
    }
  };
  // O^T += V^T P^T, V from ring slot SLOT
  auto pv = [&](auto slot_c, const bf16x8 (&p)[QG][2]) {
    constexpr int SLOT = decltype(slot_c)::value;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        lds_char* const pa = lds + kVRing + SLOT * kTileBytes + v_off[dt] + 16 * u * kRowBytes;
        const i16x4 va = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)pa);
        const i16x4 vb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(pa + 8 * kRowBytes));
        // whole-vector concatenation: element-wise assembly of the operand is mis-lowered (one dword duplicated)
        const bf16x8 vv = __builtin_bit_cast(bf16x8, __builtin_shufflevector(va, vb, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int q = 0; q < QG; ++q)
          mfma_acc(acc[q][dt], vv, p[q][u]);
      }
  };
  auto row_max = [&](const f32x16& s) -> float {
    // plain fmaxf, not v_max3 in inline asm: s comes straight from an MFMA (VGPR form), and the compiler inserts the
    // MFMA -> VALU wait states only for instructions it can see
    float mx = fmaxf(s[0], s[1]);
#pragma unroll
    for (int r = 2; r < 15; r += 2) mx = fmaxf(mx, fmaxf(s[r], s[r + 1]));
    return pair_max(fmaxf(mx, s[15]));
  };
  // all of this wave's copies but the last `keep` steps' have landed, and every wave is past its LDS reads
  auto sync_steps = [&](int keep) {
    if (keep >= 2) FVSR_WAIT_VM_LGKM0(2 * kDmaStep);
    else if (keep == 1) FVSR_WAIT_VM_LGKM0(kDmaStep);
    else FVSR_WAIT_VM_LGKM0(0);
    __builtin_amdgcn_s_barrier();
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;

  // One pass over the key tiles. MODE 0 (main): the reference m := the exact row max of the first tile (0 if it
  // has no valid key), then P = exp2(S - m); the largest partial row sum is tracked. MODE 1: row max only. MODE 2:
  // attention with m fixed to the exact row max.
  // Step T (tile T = 4b + sub, ring slot = sub): request K(T+4) and V(T+2); S(T+1) = QK(T+1); O += PV(T-1);
  // exponentials of S(T); then K(T+2) and V(T) must have landed (requested at step T-2).
  auto run = [&](auto mode_c) {
    constexpr int MODE = decltype(mode_c)::value;
#pragma unroll
    for (int q = 0; q < QG; ++q) {
      l_run[q] = 0.f;
      part_max[q] = 0.f;
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[q][d] = f32x16{};
      set_ref(q, MODE == 2 ? m_row[q] : 0.f);
      if (MODE == 1) m_row[q] = kMaskedScore;
    }
    f32x16 sA[QG], sB[QG];
    bf16x8 pA[QG][2], pB[QG][2];
    // per walked block: first-row buffer offset and keys taking part, read two blocks ahead of use
    int o0 = walk_soff(0), o1 = walk_soff(1), o2 = walk_soff(2);
    int n0 = walk_keys(0), n1 = walk_keys(1), n2 = walk_keys(2);
    int e3 = walk_entry(3);
    // prologue = virtual steps -4 .. -1: K(0..3) and V(-2..1); V(-2), V(-1) are zeros, so step 0's PV of the
    // (zero) previous P adds exact zeros
    issue_k(C0{}, o0);                issue_v(C2{}, (int)range);
    issue_k(C1{}, o0 + sub_bytes);    issue_v(C3{}, (int)range);
    issue_k(C2{}, o0 + 2 * sub_bytes); issue_v(C0{}, o0);
    issue_k(C3{}, o0 + 3 * sub_bytes); issue_v(C1{}, o0 + sub_bytes);
    sync_steps(3);   // K(0) landed
    qk(C0{}, sub_valid(n0, 0), sA);
    if (MODE == 0) {
      // reference = the exact row max of tile 0 (scaled)
#pragma unroll
      for (int q = 0; q < QG; ++q) set_ref(q, ref_of(row_max(sA[q])));
    }
#pragma unroll
    for (int q = 0; q < QG; ++q)
#pragma unroll
      for (int u = 0; u < 2; ++u) pB[q][u] = bf16x8{};
    sync_steps(1);   // K(1), K(2), V(-1), V(0) landed
    // the first LDS operands of a step (K chunk 0 of its QK tile, V^T pair 0 of its PV tile) are read at the end of
    // the step before it, so no operand read sits between the step's barrier and its first MFMA; for step 0:
    // K(1) in slot 1, V(-1) in slot 3
    bf16x8 hk;
    i16x4 hva, hvb;
    auto read_first = [&](auto kslot_c, auto vslot_c) {
      constexpr int KSL = decltype(kslot_c)::value, VSL = decltype(vslot_c)::value;
      lds_char* const pa = lds + kVRing + VSL * kTileBytes + v_off[0];
      hva = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)pa);
      hvb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(pa + 8 * kRowBytes));
      hk = *(const lds_bf16x8*)(lds + KSL * kTileBytes + k_off[0]);
    };
    if (MODE != 1) read_first(C1{}, C3{});

    // step with tile T in ring slot SUB: K(T+4) -> slot SUB, V(T+2) -> slot SUB+2, QK(T+1) <- K slot SUB+1,
    // PV(T-1) <- V slot SUB+3 (all mod 4)
    auto step = [&](auto sub_c, int valid_next, int soff_k, int soff_v, f32x16 (&s_cur)[QG], f32x16 (&s_nxt)[QG],
                    bf16x8 (&p_prev)[QG][2], bf16x8 (&p_cur)[QG][2], auto&& pre_sync) {
      constexpr int SUB = decltype(sub_c)::value;
      using KS = std::integral_constant<int, SUB>;
      using VS = std::integral_constant<int, (SUB + 2) & 3>;
      if (MODE == 1) {
        issue_k(KS{}, soff_k);
        issue_v(VS{}, soff_v);
        qk(std::integral_constant<int, (SUB + 1) & 3>{}, valid_next, s_nxt);
#pragma unroll
        for (int q = 0; q < QG; ++q) m_row[q] = fmaxf(m_row[q], row_max(s_cur[q]));
      } else {
        // 16 * QG micro-rounds with one MFMA each, fenced so the order below is the issue order, then one more for the
        // last exponential. A wave issues in order and an MFMA occupies the
        // matrix core for 32 cycles: every MFMA is followed by a slice of the other work, which issues while it runs
        // (MFMAs grouped back to back would leave that work unoverlapped). MFMA order: for c = 0..7 QK chunk c (each
        // group) and PV pair c (each group).
        // Slices: exponential I of S(T) in micro-round I (pairs packed to bf16 and summed a micro-round later); the
        // LDS operands of chunk / pair j requested up to 4 micro-rounds before use (attn_read_at); one of the step's
        // buffer->LDS copies every 4 micro-rounds.
        lds_char* const vbase = lds + kVRing + ((SUB + 3) & 3) * kTileBytes;
        lds_char* const kbase = lds + ((SUB + 1) & 3) * kTileBytes;
        i16x4 va[8], vb[8];
        bf16x8 kk[8];
        // operands of QK chunk j and PV pair j: K chunk j and V^T pair j
        auto read_ops = [&](int j) {
          if (j == 0) {   // read at the end of the step before
            va[0] = hva;
            vb[0] = hvb;
            kk[0] = hk;
            return;
          }
          lds_char* const pa = vbase + v_off[j & 3] + 16 * (j >> 2) * kRowBytes;
          va[j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)pa);
          vb[j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(pa + 8 * kRowBytes));
          kk[j] = *(const lds_bf16x8*)(kbase + k_off[j]);
        };
        auto dma = [&](auto r_c) {
          constexpr int R = decltype(r_c)::value;
          if constexpr (R < kDmaK) dma_k(KS{}, std::integral_constant<int, R>{}, soff_k);
          else dma_v(VS{}, std::integral_constant<int, R - kDmaK>{}, soff_v);
        };
        float sum[QG][2];
        float xv[2];   // the exponentials of the last two micro-rounds
        auto micro = [&](auto i_c) {
          constexpr int I = decltype(i_c)::value;
          if constexpr (I == 0) {
            read_ops(0);
            read_ops(1);
          }
          static_for<2, 8>([&](auto j_c) {
            constexpr int J = decltype(j_c)::value;
            if constexpr (attn_read_at<QG>(J) == I) read_ops(J);
          });
          if constexpr (I < 16 * QG) {
            constexpr int c = I / (2 * QG), w = I % (2 * QG);
            if constexpr (w < QG) {
              if constexpr (c > 0)
                s_nxt[w] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kk[c], qop[w][c], s_nxt[w], 0, 0, 0);
              else
                s_nxt[w] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kk[0], qop[w][0], f32x16{}, 0, 0, 0);
            } else {
              // whole-vector concatenation: element-wise assembly of the operand is mis-lowered (one dword
              // duplicated)
              const bf16x8 vv =
                  __builtin_bit_cast(bf16x8, __builtin_shufflevector(va[c], vb[c], 0, 1, 2, 3, 4, 5, 6, 7));
              mfma_acc(acc[w - QG][c & 3], vv, p_prev[w - QG][c >> 2]);
            }
          }
          // exponential I of S(T) (entry idx of group q); the exponential of the micro-round before is summed (fp32
          // sums: v_dot2 would wait for the matrix core) and, completing a pair, packed to bf16 here, a micro-round
          // after it was issued, so no wait state follows the transcendental
          if constexpr (I >= 1 && I <= 16 * QG) {
            constexpr int J = I - 1, qj = J >> 4, ij = J & 15;
            if constexpr (ij < 2) sum[qj][ij] = xv[J & 1];
            else sum[qj][ij & 1] += xv[J & 1];
            if constexpr ((J & 1) == 1) {
              p_cur[qj][ij >> 3][(ij & 7) - 1] = (bf16)xv[0];
              p_cur[qj][ij >> 3][ij & 7] = (bf16)xv[1];
              // the pair is packed here, in this micro-round: without a use before the reference check the
              // compiler sinks the packs past it (the raise recomputes them) into the step's tail
              const u32x4 pw = __builtin_bit_cast(u32x4, p_cur[qj][ij >> 3]);
              asm volatile("" ::"v"(pw[(ij & 7) >> 1]));
            }
          }
          if constexpr (I < 16 * QG) {
            constexpr int q = I >> 4, idx = I & 15;
            xv[I & 1] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[q][idx], c_scale, negm[q]));
          }
          if constexpr ((I & 3) == 1 && I / 4 < kDmaStep) dma(std::integral_constant<int, I / 4>{});
          if constexpr (I == 16 * QG)
            read_first(std::integral_constant<int, (SUB + 2) & 3>{}, std::integral_constant<int, SUB>{});
          __builtin_amdgcn_sched_barrier(0);
        };
        static_for<0, 16 * QG + 1>(micro);
        float part[QG];
        bool grow = false;
#pragma unroll
        for (int q = 0; q < QG; ++q) {
          part[q] = sum[q][0] + sum[q][1];
          grow |= !(part[q] <= kGrowSum);   // either half of a row; also inf / NaN
        }
        if (__ballot(grow) != 0) {
          // raise the reference of the rows that grew to their max in S(T); the other rows keep theirs (their
          // scale is 1 and every operation below is exact and changes nothing)
          acc_drain();
#pragma unroll
          for (int q = 0; q < QG; ++q) {
            const bool gq = !(pair_max(part[q]) <= kGrowSum);
            const float m_new = gq ? row_max(s_cur[q]) * c_scale : m_ref[q];
            const float sc = __builtin_amdgcn_exp2f(m_ref[q] - m_new);
            set_ref(q, m_new);
            float t[2] = {0.f, 0.f};
#pragma unroll
            for (int idx = 1; idx < 16; idx += 2) {
              const float x0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[q][idx - 1], c_scale, negm[q]));
              const float x1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[q][idx], c_scale, negm[q]));
              p_cur[q][idx >> 3][(idx & 7) - 1] = (bf16)x0;
              p_cur[q][idx >> 3][idx & 7] = (bf16)x1;
              t[(idx >> 1) & 1] += x0 + x1;
            }
            part[q] = t[0] + t[1];
            l_run[q] *= sc;
            part_max[q] *= sc;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
              for (int i = 0; i < 16; ++i) acc[q][dt][i] *= sc;
          }
        }
#pragma unroll
        for (int q = 0; q < QG; ++q) {
          l_run[q] += part[q];
          part_max[q] = fmaxf(part_max[q], part[q]);
        }
        // last in the step: a branch before the row sums would let the compiler sink the exponentials past it
        if (valid_next < kTileKeys) {
#pragma unroll
          for (int q = 0; q < QG; ++q) mask_tile(s_nxt[q], valid_next);
        }
      }
      // keep every instruction of this step on its side of the barrier; the copies of the step before have landed
      // (the next step's first operands, read above, were waited for one step earlier)
      __builtin_amdgcn_sched_barrier(0);
      pre_sync();
      sync_steps(1);
      __builtin_amdgcn_sched_barrier(0);
    };
    for (int b = 0; b < nblocks; ++b) {
      const int o3 = entry_soff(b + 3, e3), n3 = entry_keys(b + 3, e3);
      // step 4b+s: QK tile 4b+s+1, K tile 4b+s+4 (block b+1), V tile 4b+s+2
      auto nop = [] {};
      step(C0{}, sub_valid(n0, 1), o1, o0 + 2 * sub_bytes, sA, sB, pB, pA, nop);
      step(C1{}, sub_valid(n0, 2), o1 + sub_bytes, o0 + 3 * sub_bytes, sB, sA, pA, pB, nop);
      step(C2{}, sub_valid(n0, 3), o1 + 2 * sub_bytes, o1, sA, sB, pB, pA, nop);
      // the next block's list entry loads right before the step's wait, which absorbs it
      step(C3{}, sub_valid(n1, 0), o1 + 3 * sub_bytes, o1 + sub_bytes, sB, sA, pA, pB,
           [&] { e3 = walk_entry(b + 4); });
      o0 = o1; o1 = o2; o2 = o3;
      n0 = n1; n1 = n2; n2 = n3;
    }
    if (MODE != 1) {
      pv(C3{}, pB);   // PV of the last tile (4 * nblocks - 1, slot 3)
      acc_drain();
    }
    // drain the zero-fill copies requested past the end before LDS is reused
    FVSR_WAIT_VM_LGKM0(0);
    __builtin_amdgcn_s_barrier();
  };

  run(std::integral_constant<int, 0>{});
  // rows whose exponentials all underflowed (the reference came from a tile with no valid key and every score is
  // far below it): redo the workgroup exactly (row max pass, then attention with that max); workgroup-uniform so the
  // barriers match
  {
    bool bad = false;
#pragma unroll
    for (int q = 0; q < QG; ++q) bad |= !(pair_max(part_max[q]) >= 2.3283064e-10f);
    int* flag = (int*)smem;
    if (tid == 0) flag[0] = 0;
    __syncthreads();
    if (__ballot(bad) != 0 && lane == 0) flag[0] = 1;
    __syncthreads();
    const bool redo = flag[0] != 0;
    __syncthreads();
    if (redo) {
      run(std::integral_constant<int, 1>{});
#pragma unroll
      for (int q = 0; q < QG; ++q) m_row[q] = ref_of(m_row[q]);
      run(std::integral_constant<int, 2>{});
    }
  }

#pragma unroll
  for (int q = 0; q < QG; ++q) attn_store<DIRECT, bf16>(a, it, wave * QG + q, acc[q], m_ref[q], pair_sum(l_run[q]), O);
  if constexpr (DIRECT) break;
  }   // next item
}

// Rows (head, query block) for the persistent bf16 walk, and the per-XCD queue counters. One workgroup. First a
// counting sort by decreasing key-list length in 255 bins of ceil(longest / 255) blocks (exact lengths up to 255
// blocks). Then every wave of `grid` consecutive items of that order (one
// item per workgroup) is re-sorted by row id (head-major, neighbouring query blocks together) and dealt so that XCD x
// (workgroups b with b % 8 == x, dispatch is round-robin over the XCDs) holds positions x, x + 8, .. of the wave:
// one contiguous range of rows, whose key lists overlap, so the XCD's L2 serves the key blocks they share.
// next_dealt_item hands the positions out per XCD. The order does not affect results. Scans are wave-wide
// (shuffles) with one step across the waves. Up to kOrderLdsRows rows the lengths' bins and the sorted order stay in
// LDS (kcnt is read once, the dealt order written once) and, while the waves' bitmaps fit together, every wave is
// ranked in one pass (one bitmap segment per wave, one scan); beyond, the sorted order is staged in `order` itself
// and the waves are ranked one after another. When every list has the same length the row-id order is such an order
// already and is dealt as it stands.
constexpr int kOrderLdsRows = 8192;
__global__ __launch_bounds__(1024) void attn_order_kernel(const int32_t* __restrict__ kcnt, int rows, int nk_stride,
                                                          int grid, int32_t* __restrict__ order,
                                                          int32_t* __restrict__ counters) {
  constexpr int kBins = 256;
  constexpr int kWords = 4096;   // row-id bitmap words: the bitmap rank serves up to 32 x 4096 rows
  __shared__ int bin_start[kBins];
  __shared__ int wtot[16];
  __shared__ __attribute__((aligned(16))) int first[kMaxPersistentWgs];   // one wave; padded with INT_MAX
  __shared__ unsigned bm[kWords];
  __shared__ int wpre[kWords];                                            // set bits in the words before word w
  __shared__ int lord[kOrderLdsRows];                                     // the sorted order (rows <= kOrderLdsRows)
  __shared__ uint8_t lbin[kOrderLdsRows];                                 // each row's bin (rows <= kOrderLdsRows)
  __shared__ int s_longest, s_mixed;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool in_lds = rows <= kOrderLdsRows;
  int* const sorted = in_lds ? lord : order;
  if (tid < kBins) bin_start[tid] = 0;
  if (tid == 0) {
    s_longest = 0;
    s_mixed = 0;
  }
  __syncthreads();
  auto list_len = [&](int r) -> int { return max(0, min(kcnt[r], nk_stride)); };
  // the longest list, and whether the lengths differ at all (the lengths wait in lord until the sort overwrites it);
  // a thread's loads are issued together, so their latencies overlap
  {
    const int c0 = list_len(0);
    int m = 0;
    bool mixed = false;
    for (int r0 = tid; r0 < rows; r0 += 4 * 1024) {
      int c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = list_len(min(r0 + u * 1024, rows - 1));   // loads without branches
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (r0 + u * 1024 < rows) {
          if (in_lds) lord[r0 + u * 1024] = c[u];
          m = max(m, c[u]);
          mixed |= c[u] != c0;
        }
      }
    }
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
    if (lane == 0) atomicMax(&s_longest, m);
    if (__ballot(mixed) != 0 && lane == 0) s_mixed = 1;
  }
  __syncthreads();
  // every list of one length (the cross-attention's lists): the row-id order is already
  // sorted by length and each of its waves by row id, so the sort and the ranking are skipped and the rows are dealt
  // where they stand
  const bool one_len = s_mixed == 0;
  if (!one_len) {
    const int width = max(1, (s_longest + kBins - 2) / (kBins - 1));   // blocks per bin
    auto bin_len = [&](int c) -> int {   // bin 0 = the longest lists
      const int len = c <= 0 ? 0 : min((c + width - 1) / width, kBins - 1);
      return kBins - 1 - len;
    };
    auto bin_of = [&](int r) -> int { return bin_len(list_len(r)); };
    for (int r = tid; r < rows; r += 1024) {
      const int bn = in_lds ? bin_len(lord[r]) : bin_of(r);
      if (in_lds) lbin[r] = (uint8_t)bn;
      atomicAdd(&bin_start[bn], 1);
    }
    __syncthreads();
    // exclusive scan of the 256 bin counts by waves 0..3
    {
      const int v = tid < kBins ? bin_start[tid] : 0;
      const int incl = (int)wave_incl_scan((unsigned)v);
      if (tid < kBins && lane == 63) wtot[wave] = incl;
      __syncthreads();
      if (tid < kBins) {
        int base = 0;
        for (int w = 0; w < wave; ++w) base += wtot[w];
        bin_start[tid] = base + incl - v;
      }
    }
    __syncthreads();
    for (int r = tid; r < rows; r += 1024) sorted[atomicAdd(&bin_start[in_lds ? (int)lbin[r] : bin_of(r)], 1)] = r;
  }
  __threadfence_block();
  __syncthreads();
  grid = min(grid, kMaxPersistentWgs);
  // position p of the sorted order goes to wave p / grid; XCD x holds m_x = (nw - x + 7) / 8 positions x, x + 8, ..
  // of a wave of nw items, and ranks s_x .. s_x + m_x - 1 (by row id) go to it
  auto deal = [&](int w0, int nw, int rank, int r) {
    int x = 0, s0 = 0;
    while (s0 + (nw - x + kXcds - 1) / kXcds <= rank) {
      s0 += (nw - x + kXcds - 1) / kXcds;
      ++x;
    }
    order[w0 + (rank - s0) * kXcds + x] = r;
  };
  // exclusive scan of the popcounts of bm[0 .. n) into wpre (4 words per thread, n <= kWords)
  auto scan_words = [&](int n) {
    int c[4], csum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int w = 4 * tid + i;
      c[i] = w < n ? __popc(bm[w]) : 0;
      csum += c[i];
    }
    const int incl = (int)wave_incl_scan((unsigned)csum);
    if (lane == 63) wtot[wave] = incl;
    __syncthreads();
    int run = incl - csum;
    for (int w = 0; w < wave; ++w) run += wtot[w];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (4 * tid + i < n) wpre[4 * tid + i] = run;
      run += c[i];
    }
    __syncthreads();
  };
  const int rwords = (rows + 31) / 32;
  const int nwaves = (rows + grid - 1) / grid;
  if (one_len) {
    for (int p = tid; p < rows; p += 1024) {
      const int w0 = p / grid * grid;
      deal(w0, min(grid, rows - w0), p - w0, p);
    }
  } else if (in_lds && nwaves * rwords <= kWords) {
    // every wave at once: wave w's rows set their bits in bitmap segment w, one scan covers all segments
    for (int i = tid; i < nwaves * rwords; i += 1024) bm[i] = 0u;
    __syncthreads();
    for (int p = tid; p < rows; p += 1024) {
      const int r = sorted[p];
      atomicOr(&bm[(p / grid) * rwords + (r >> 5)], 1u << (r & 31));
    }
    __syncthreads();
    scan_words(nwaves * rwords);
    for (int p = tid; p < rows; p += 1024) {
      const int r = sorted[p], w = p / grid, wi = w * rwords + (r >> 5);
      const int rank = wpre[wi] - wpre[w * rwords] + __popc(bm[wi] & ((1u << (r & 31)) - 1u));
      deal(w * grid, min(grid, rows - w * grid), rank, r);
    }
  } else {
    const bool use_bitmap = rows <= kWords * 32;
    const int words = use_bitmap ? rwords : 0;
    for (int w0 = 0; w0 < rows; w0 += grid) {
      const int nw = min(grid, rows - w0);
      for (int i = tid; i < kMaxPersistentWgs; i += 1024) first[i] = i < nw ? sorted[w0 + i] : 0x7fffffff;
      for (int w = tid; w < words; w += 1024) bm[w] = 0u;
      __syncthreads();
      // rank of each row of the wave among them by row id: a bitmap over the row ids and a scan of its per-word
      // popcounts; beyond 32 x 4096 rows, a scan of the wave's rows themselves
      if (use_bitmap) {
        for (int i = tid; i < nw; i += 1024) atomicOr(&bm[first[i] >> 5], 1u << (first[i] & 31));
        __syncthreads();
        scan_words(words);
      }
      const int n4 = (nw + 31) / 32 * 8;   // int4 groups to scan, a multiple of the unroll
      for (int i = tid; i < nw; i += 1024) {
        const int r = first[i];
        int rank = 0;   // rows are distinct: ranks are a permutation of 0 .. nw - 1
        if (use_bitmap) {
          rank = wpre[r >> 5] + __popc(bm[r >> 5] & ((1u << (r & 31)) - 1u));
        } else {
#pragma unroll 8
          for (int j = 0; j < n4; ++j) {
            const int4 f = reinterpret_cast<const int4*>(first)[j];
            rank += (f.x < r) + (f.y < r) + (f.z < r) + (f.w < r);
          }
        }
        deal(w0, nw, rank, r);
      }
      __syncthreads();
    }
  }
  // queue y's counter starts past the first wave (the workgroups take it without the counters)
  if (tid < kXcds) counters[8 * tid] = (grid - tid + kXcds - 1) / kXcds;
}

// ------------------------------------------------------------------------------------------------------------
// fp32 (parity lane)
// ------------------------------------------------------------------------------------------------------------
// The products run on the bf16 matrix cores: every fp32 operand is the exact sum of three bf16 parts (24 significand
// bits = 8 + 8 + 8, each part the rounded remainder of the ones before it), and a product takes the six partial
// products above 2^-24 of it, smallest first, accumulated in fp32. The three left out (m l, l m, l l) are 2^-26 of the
// product at most, below the rounding of the fp32 sum. bf16 has fp32's exponents, so no operand is scaled by its
// neighbours and the error of a product is relative to that product, whatever else the list holds. Six k = 16 products
// cost 192 matrix-core cycles per 32 x 32 x 16 block of products, against 512 for the eight k = 2 fp32 ones. (Two fp16 parts
// and three products would cost 96, but fp16 holds 2^-24 .. 65504 only: under any scale shared by a row, a tile or a
// list, elements far below the largest lose their bits, also where the largest has no weight in the result.)
//
// At the ends of the range:
//   magnitudes above 2^59 (infinities among them): the walk stops and the item is computed on the fp32 matrix instructions
//      (f32_exact_walk; 576 rows x 24 blocks with one such key a block 1750 us, where the split takes 630 without them, a whole
//      walk before the exact one 2300 and a kernel for these instructions alone 1184). Up to there no partial product or sum
//      of a score that fp32 holds overflows.
//   V is multiplied by 2^24 before the split, so that every part of the smallest fp32 number is a normal bf16; the
//      output takes the power back, exactly. Parts of Q and K below 2^-126 may be lost: at most 2^-126 2^59 128 = 2^-60 of a
//      score, an absolute error that the exponential does not see.
// NaNs propagate through the parts.
//
// A workgroup = 4 wave64s x 32 queries, two per CU (48 KB of tile LDS, at most 256 registers a wave), so that one
// workgroup's softmax and waits run under the other's products. Keys stream in tiles of 32: a tile's fp32 rows are
// loaded into registers a phase ahead (raw buffer loads, rows past the buffer read 0), split once per workgroup and
// stored as three bf16 planes with the 16-byte chunk swizzles of the bf16 walk. K and V planes have one buffer each (two
// would leave one workgroup a CU): V(T) is split and stored between the products of the scores of tile T, K(T+1) between
// those of its output, with a barrier after each. S^T = K Q^T leaves each lane one query's scores; the lazy online softmax
// is in fp32, and P is split in registers.
//
// Bound by the matrix cores: 504 rows x 32 blocks 651 us, 208 TFLOP/s of fp32 products, where six bf16 products at the
// rate of a large bf16 GEMM would give 228; the splits, the softmax and the operand reads (about 500 VALU and 96 LDS
// instructions a wave and tile) run under the 96 MFMAs (3072 cycles). 512 x 512, 12 heads, us on the fp32 instructions
// and now: layer call of 2 latent frames over 6 311, 130; two-chunk clip 3841, 1270 (two scaled fp16 parts: 101 and 838, wrong
// for the unequal operands named above). Its error against 64 bits is the smallest of the three: 8.1e-7, 3.8e-7 (fp16
// parts 3.8e-7) and 1.9e-6, 8.7e-7 (1.1e-6).
constexpr int kF32Plane = kTileBytes;              // one bf16 plane of a 32-key tile
constexpr float kSplitMax = 5.7646075e17f;         // 2^59: the largest magnitude the split serves
constexpr float kSplitV = 16777216.f;              // 2^24: V's factor before the split
constexpr int kExactLd = 132;                      // padded fp32 row of the exact walk's tiles (floats)

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;

// two values as their packed bf16 parts h + m + l
__device__ __forceinline__ void split_pair(float a, float b, unsigned& h, unsigned& m, unsigned& l) {
  auto pack = [](float x, float y) -> unsigned {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{x, y}, bf16x2));
  };
  auto lo = [](unsigned u) { return __uint_as_float(u << 16); };
  auto hi = [](unsigned u) { return __uint_as_float(u & 0xffff0000u); };
  h = pack(a, b);
  const float ra = a - lo(h), rb = b - hi(h);
  m = pack(ra, rb);
  l = pack(ra - lo(m), rb - hi(m));
}

// partial product N (0 .. 5, smallest first) of a k = 16 step: A's parts ah, am, al by B's bh, bm, bl
template <int N>
__device__ __forceinline__ void mfma_part(f32x16& acc, const bf16x8& ah, const bf16x8& am, const bf16x8& al,
                                          const bf16x8& bh, const bf16x8& bm, const bf16x8& bl) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(N == 0 ? al : N == 2 || N == 3 ? am : ah,
                                                N == 1 ? bl : N == 2 || N == 4 ? bm : bh, acc, 0, 0, 0);
}

// One item on the fp32 matrix cores (v_mfma_f32_32x32x2_f32), for operands the split cannot hold. Every wave of the
// workgroup calls it together; smem holds 2 x 32 x kExactLd floats. Same lazy softmax and output layout as the kernel.
__device__ __forceinline__ void f32_exact_walk(const AttnArgs& a, int h, int64_t qrow,
                                                         const int32_t* __restrict__ klist, int nblocks, float* smem,
                                                         f32x16 (&acc_o)[4], float& m_run, float& l_run) {
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const float* __restrict__ Q = (const float*)a.q + h * kHeadDim;
  const float* __restrict__ K = (const float*)a.k + h * a.kv_head_stride;
  const float* __restrict__ V = (const float*)a.v + h * a.kv_head_stride;
  float* const ks = smem;
  float* const vs = smem + kTileKeys * kExactLd;
  m_run = -INFINITY;
  l_run = 0.f;
#pragma unroll
  for (int d = 0; d < 4; ++d) acc_o[d] = f32x16{};
  for (int T = 0; T < 4 * nblocks; ++T) {
    const int j = klist[T >> 2], sub = T & 3;
    const int64_t valid = (unsigned)j < (unsigned)a.nk ? a.lk - ((int64_t)j * kBlock + sub * kTileKeys) : 0;
    const int64_t row0 = valid > 0 ? a.map.row(j) + sub * kTileKeys : 0;
    __syncthreads();   // the tile before has been read
    for (int e = tid; e < kTileKeys * 32; e += 256) {
      const int r = e >> 5, c4 = (e & 31) * 4;
      f32x4 kv = f32x4{0, 0, 0, 0}, vv = f32x4{0, 0, 0, 0};
      if (r < valid) {
        kv = *(const f32x4*)(K + (row0 + r) * a.kv_ld + c4);
        vv = *(const f32x4*)(V + (row0 + r) * a.kv_ld + c4);
      }
      *(f32x4*)(ks + r * kExactLd + c4) = kv;
      *(f32x4*)(vs + r * kExactLd + c4) = vv;
    }
    __syncthreads();
    f32x16 s = f32x16{};
    for (int i = 0; i < 16; ++i) {
      const f32x4 kf = *(const f32x4*)(ks + l32 * kExactLd + 8 * i + 4 * g);
      f32x4 qf = f32x4{0, 0, 0, 0};
      if (qrow < a.lq) qf = *(const f32x4*)(Q + qrow * a.ld + 8 * i + 4 * g);
#pragma unroll
      for (int b = 0; b < 4; ++b) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[b], qf[b], s, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (8 * (r >> 2) + 4 * g + (r & 3) >= valid) s[r] = -INFINITY;
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    const float m_use = rescale_if_grown<4>(pair_max(mx) * a.c, m_run, l_run, acc_o);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], a.c, -m_use));
      l_run += s[r];
    }
    // k-step r pairs key 8(r/4) + 4g + r%4 (this lane's P entry r) with k-index g
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = 8 * (r >> 2) + 4 * g + (r & 3);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vs[key * kExactLd + 32 * dt + l32], s[r], acc_o[dt], 0, 0, 0);
    }
  }
}

template <bool DIRECT>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 2)))
void attn_f32_kernel(AttnArgs a, const int32_t* __restrict__ kidx, const int32_t* __restrict__ kcnt,
                     const float* __restrict__ Q, float* __restrict__ O, int32_t* __restrict__ order,
                     int32_t* __restrict__ counter) {
  __shared__ __attribute__((aligned(1024))) char smem[6 * kF32Plane];   // K planes h, m, l, then V planes h, m, l
  static_assert(sizeof(float) * 2 * kTileKeys * kExactLd <= 6 * kF32Plane, "the exact walk's tiles fit");
  __shared__ int item_s;
  __shared__ int huge_s;   // a magnitude above kSplitMax was met: the walk stops after the block

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  const int rows = a.heads * a.nq;
  const uint32_t row_bytes = (uint32_t)a.kv_ld * 4;
  const uint32_t range = (uint32_t)a.kv_bytes;
  __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void*)a.k, 0, range, 0x00020000);
  __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)a.v, 0, range, 0x00020000);
  // staging: this thread loads 8 floats of rows r_ld and r_ld + 16 of a tile, one 16-byte chunk of each plane
  const int r_ld = tid >> 4, c_ld = tid & 15;
  const int st_k[2] = {r_ld * kRowBytes + ((c_ld ^ swz_k(r_ld)) << 4),
                       (r_ld + 16) * kRowBytes + ((c_ld ^ swz_k(r_ld + 16)) << 4)};
  const int st_v[2] = {r_ld * kRowBytes + ((c_ld ^ swz_v(r_ld)) << 4),
                       (r_ld + 16) * kRowBytes + ((c_ld ^ swz_v(r_ld + 16)) << 4)};
  // operand reads, as in the bf16 walk
  // (chunk 2 t + g of a K row is 32 t xor chunk g's offset, V columns 32 dt .. are 64 dt xor columns 0 ..'s)
  const int k_off = l32 * kRowBytes + ((g ^ swz_k(l32)) << 4);
  const int G = lane >> 4, mm = lane & 15, vr = 4 * (G >> 1) + (mm >> 2);
  const int v_off = vr * kRowBytes + (((2 * (G & 1) + ((mm & 3) >> 1)) ^ swz_v(vr)) << 4) + (mm & 1) * 8;
  lds_char* const lds = (lds_char*)(uintptr_t)lds_addr(smem);
  lds_char* const ldsv = lds + 3 * kF32Plane;

  for (bool first = true;; first = false) {
    AttnItem it;
    if (!next_item<DIRECT, 256>(a, kcnt, order, counter, rows, first, tid, &item_s, (int*)smem, it)) break;
    if (it.nblocks <= 0) {
      attn_empty_item<float>(a, it, O, tid, 256);
      if constexpr (DIRECT) break;
      else continue;
    }
    const int32_t* __restrict__ klist = kidx + (int64_t)it.row * a.nk_stride + it.b0;
    const int nblocks = it.nblocks;
    const int64_t qrow = (int64_t)it.qb * kBlock + wave * 32 + l32;

    // walked block b: byte offset of its first row (past the buffer for an index outside [0, nk) and past the walk's end)
    // and its keys taking part
    auto walk_entry = [&](int b) -> int { return b < nblocks ? klist[b] : -1; };
    auto entry_off = [&](int j) -> uint32_t {
      return (unsigned)j < (unsigned)a.nk ? (uint32_t)a.map.row(j) * row_bytes : range;
    };
    auto entry_keys = [&](int j) -> int {
      return (unsigned)j < (unsigned)a.nk ? (int)min<int64_t>(kBlock, a.lk - (int64_t)j * kBlock) : 0;
    };
    const uint32_t sub_bytes = kTileKeys * row_bytes;
    const uint32_t ld_off = r_ld * row_bytes + (uint32_t)(it.h * a.kv_head_stride * 4) + c_ld * 32;
    f32x4 raw[4];   // this thread's part of the K or V tile to be split next
    // half I: the 8 floats of row r_ld + 16 I. The sum stays below 2^32: a listed block's offset and the head's lie inside
    // the buffer (< 2^31 bytes), the offset past it is the buffer's size.
    auto load_half = [&](__amdgpu_buffer_rsrc_t rs, auto i_c, uint32_t off) {
      constexpr int I = decltype(i_c)::value;
      const uint32_t o = ld_off + off + I * 16 * row_bytes;
      raw[2 * I] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
      raw[2 * I + 1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, o + 16, 0, 0));
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;

    float mag = 0.f;   // largest magnitude this thread split
    // Q as the B operand of S^T = K Q^T
    bf16x8 qh[8], qm[8], ql[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      f32x4 x[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
      if (qrow < a.lq) {
        const float* p = Q + qrow * a.ld + it.h * kHeadDim + 16 * t + 8 * g;
        x[0] = *(const f32x4*)p;
        x[1] = *(const f32x4*)(p + 4);
      }
      u32x4 h, m, l;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = x[i >> 1][2 * (i & 1)], r = x[i >> 1][2 * (i & 1) + 1];
        unsigned hw, mw, lw;
        split_pair(p, r, hw, mw, lw);
        mag = fmaxf(mag, fmaxf(fabsf(p), fabsf(r)));
        h[i] = hw;
        m[i] = mw;
        l[i] = lw;
      }
      qh[t] = __builtin_bit_cast(bf16x8, h);
      qm[t] = __builtin_bit_cast(bf16x8, m);
      ql[t] = __builtin_bit_cast(bf16x8, l);
    }

    // pair I (elements 2 I, 2 I + 1 of this thread's 16) of the raw tile, times `scale`; after every other pair half a chunk
    // is stored at its place of the planes (chunks of rows r_ld and r_ld + 16 at at[0] and at[1])
    u32x2 wh, wm, wl;
    auto split_raw = [&](auto i_c, float scale, lds_char* planes, const int (&at)[2]) {
      constexpr int I = decltype(i_c)::value;
      const float x = raw[I >> 1][2 * (I & 1)], y = raw[I >> 1][2 * (I & 1) + 1];
      unsigned hw, mw, lw;
      split_pair(x * scale, y * scale, hw, mw, lw);
      mag = fmaxf(mag, fmaxf(fabsf(x), fabsf(y)));
      asm volatile("" : "+v"(mag));   // here: the compiler would keep the elements of a whole block for one late maximum
      wh[I & 1] = hw;
      wm[I & 1] = mw;
      wl[I & 1] = lw;
      if constexpr ((I & 1) == 1) {
        lds_char* const to = planes + at[I >> 2] + (I & 2) * 4;
        *(lds_u32x2*)to = wh;
        *(lds_u32x2*)(to + kF32Plane) = wm;
        *(lds_u32x2*)(to + 2 * kF32Plane) = wl;
      }
    };

    f32x16 acc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[d] = f32x16{};
    float m_run = -INFINITY, l_run = 0.f;

    // One tile: K is stored, V waits in raw; the next tile is at byte offset off1. 48 rounds of one MFMA each for the
    // scores, then 48 for the output, fenced so that the order below is the issue order: a wave issues in order and an MFMA
    // holds the matrix core for 32 cycles, so a slice of the other work follows each. V is split under the scores, K of the
    // next tile and the second half of P under the output; raw's halves are requested anew as they are split.
    auto step = [&](int valid, uint32_t off1) {
      bf16x8 kh[8], km[8], kl[8];
      auto read_k = [&](int plane, int t) -> bf16x8 {
        return *(const lds_bf16x8*)(lds + plane * kF32Plane + (k_off ^ (t << 5)));
      };
      kl[0] = read_k(2, 0);
      kh[0] = read_k(0, 0);
      km[0] = read_k(1, 0);
      f32x16 s = f32x16{};
      // the five small products of every chunk first, then the large ones: only these round at the score's own size
      static_for<0, 48>([&](auto r_c) {
        constexpr int r = decltype(r_c)::value, t = r < 40 ? r / 5 : r - 40, n = r < 40 ? r % 5 : 5;
        // the next chunk's parts, each as late as its latency allows: l and m into the registers that their last use freed
        if constexpr (r < 40) {
          if constexpr (n == 1 && t + 1 < 8) kl[t + 1] = read_k(2, t + 1);
          if constexpr (n == 2) kh[(t + 1) & 7] = read_k(0, (t + 1) & 7);
          if constexpr (n == 3 && t + 1 < 8) km[t + 1] = read_k(1, t + 1);
          if constexpr (n == 4 && t == 7) kh[1] = read_k(0, 1);
        } else if constexpr (t + 2 < 8) {
          kh[t + 2] = read_k(0, t + 2);
        }
        mfma_part<n>(s, kh[t], km[t], kl[t], qh[t], qm[t], ql[t]);
        if constexpr (r % 6 == 3) split_raw(std::integral_constant<int, r / 6>{}, kSplitV, ldsv, st_v);
        if constexpr (r == 22) load_half(krs, I0{}, off1);
        if constexpr (r == 46) load_half(krs, I1{}, off1);
        __builtin_amdgcn_sched_barrier(0);
      });
      __syncthreads();   // K has been read, V is stored
      bf16x8 vh[8], vm[8], vl[8];
      auto read_v = [&](int plane, int i) -> bf16x8 {   // i = 4 u + dt: V^T operand of keys 16 u .., dims 32 dt ..
        lds_char* const pa = ldsv + plane * kF32Plane + (v_off ^ ((i & 3) << 6)) + 16 * (i >> 2) * kRowBytes;
        const i16x4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)pa);
        const i16x4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(pa + 8 * kRowBytes));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7));
      };
      vl[0] = read_v(2, 0);
      vh[0] = read_v(0, 0);
      vm[0] = read_v(1, 0);
      if (valid < kTileKeys) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + 4 * g + (r & 3) >= valid) s[r] = -INFINITY;
      }
      float mx = fmaxf(s[0], s[1]);
#pragma unroll
      for (int r = 2; r < 16; ++r) mx = fmaxf(mx, s[r]);
      const float m_use = rescale_if_grown<4>(pair_max(mx) * a.c, m_run, l_run, acc);
      u32x4 ph[2], pm[2], pl[2];
      float px, py, sum[2] = {0.f, 0.f};
      auto exp_x = [&](int j) { px = __builtin_amdgcn_exp2f(fmaf(s[2 * j], a.c, -m_use)); };
      auto exp_y = [&](int j) { py = __builtin_amdgcn_exp2f(fmaf(s[2 * j + 1], a.c, -m_use)); };
      auto split_p = [&](int j) {   // keys 2 j, 2 j + 1 of this lane's 16
        sum[0] += px;
        sum[1] += py;
        asm volatile("" : "+v"(sum[0]), "+v"(sum[1]));   // here: summed later, all 16 would stay in registers
        unsigned hw, mw, lw;
        split_pair(px, py, hw, mw, lw);
        ph[j >> 2][j & 3] = hw;
        pm[j >> 2][j & 3] = mw;
        pl[j >> 2][j & 3] = lw;
      };
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        exp_x(j);
        exp_y(j);
        split_p(j);
      }
      __builtin_amdgcn_sched_barrier(0);
      // O^T += V^T P^T
      static_for<0, 48>([&](auto r_c) {
        constexpr int r = decltype(r_c)::value, i = r / 6, u = i / 4, n = r % 6;
        if constexpr (i + 1 < 8) {
          if constexpr (n == 1) vl[i + 1] = read_v(2, i + 1);
          if constexpr (n == 2) vh[i + 1] = read_v(0, i + 1);
          if constexpr (n == 4) vm[i + 1] = read_v(1, i + 1);
        }
        mfma_part<n>(acc[i & 3], vh[i], vm[i], vl[i], __builtin_bit_cast(bf16x8, ph[u]),
                     __builtin_bit_cast(bf16x8, pm[u]), __builtin_bit_cast(bf16x8, pl[u]));
        if constexpr (u == 0) {
          if constexpr (n == 1) exp_x(4 + i);
          if constexpr (n == 2) exp_y(4 + i);
          if constexpr (n == 4) split_p(4 + i);
        }
        if constexpr (n == 3) split_raw(std::integral_constant<int, i>{}, 1.f, lds, st_k);
        if constexpr (r == 22) load_half(vrs, I0{}, off1);
        if constexpr (r == 46) load_half(vrs, I1{}, off1);
        __builtin_amdgcn_sched_barrier(0);
      });
      l_run += sum[0] + sum[1];
      __syncthreads();   // V has been read, K of the next tile is stored
    };

    int e0 = walk_entry(0), e1 = walk_entry(1);
    uint32_t o0 = entry_off(e0);
    auto sub_off = [&](uint32_t o, int sub) -> uint32_t { return o == range ? range : o + sub * sub_bytes; };
    load_half(krs, I0{}, o0);
    load_half(krs, I1{}, o0);
    static_for<0, 8>([&](auto i_c) { split_raw(i_c, 1.f, lds, st_k); });
    load_half(vrs, I0{}, o0);
    load_half(vrs, I1{}, o0);
    if (tid == 0) huge_s = 0;
    __syncthreads();   // K is stored
    for (int b = 0; b < nblocks; ++b) {
      const int n0 = entry_keys(e0);
      const uint32_t o1 = entry_off(e1);
      e0 = e1;
      e1 = walk_entry(b + 2);
#pragma nounroll   // one copy of the step: it fills the instruction cache
      for (int sub = 0; sub < 4; ++sub) {
        if (sub == 2 && !(mag <= kSplitMax)) huge_s = 1;   // barriers on both sides: every wave reads the same below
        step(n0 - sub * kTileKeys, sub_off(sub < 3 ? o0 : o1, (sub + 1) & 3));
      }
      if (huge_s != 0) break;
      o0 = o1;
    }
    if (__syncthreads_or(!(mag <= kSplitMax))) {
      f32_exact_walk(a, it.h, qrow, klist, nblocks, (float*)smem, acc, m_run, l_run);
    } else {
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[d][r] *= 1.f / kSplitV;
    }
    attn_store<DIRECT, float>(a, it, wave, acc, m_run == -INFINITY ? 0.f : m_run, pair_sum(l_run), O);
    if constexpr (DIRECT) break;
    __syncthreads();   // smem and item_s are free for the next item
  }
}

// ------------------------------------------------------------------------------------------------------------
// merge of split rows
// ------------------------------------------------------------------------------------------------------------
// O of a row split into pieces: sum_p 2^(m_p - M) acc_p / sum_p 2^(m_p - M) l_p, M the largest reference of the pieces
// with a weight. Pieces of one count have their results `rows` apart, those of split_item one after another (plan: n << 16 |
// the first piece's number; rows of one piece are written already). One workgroup per 32
// queries of a row, one wave per 32 dims; reads 64 KB a piece and row in register order, so it runs at the rate the
// partial results come out of the caches.
template <typename T>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnArgs a, const int32_t* __restrict__ plan, T* __restrict__ O) {
  typedef T Tx4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, g = lane >> 5, l32 = lane & 31, dt = threadIdx.x >> 6;
  const int row = blockIdx.x >> 2, group = blockIdx.x & 3;
  const int rows = a.heads * a.nq;
  const bool planned = a.split_items > 0;
  const int pieces = planned ? plan[row] >> 16 : a.pieces, first = planned ? plan[row] & 0xffff : row;
  if (pieces <= 1) return;
  const int listed = planned ? 0 : min(a.kcnt[row], a.nk_stride);
  const int h = row / a.nq, qb = row - h * a.nq;
  const float* const ml = a.part_ml + (int64_t)first * 2 * kBlock + group * 32 + l32;
  const float* const po = a.part_o + ((int64_t)first * 4 + group) * (32 * kHeadDim) + 1024 * dt + 4 * lane;
  const int64_t ml_step = (int64_t)(planned ? 1 : rows) * 2 * kBlock;   // piece to piece
  const int64_t o_step = (int64_t)(planned ? 1 : rows) * kBlock * kHeadDim;
  float M = -INFINITY;
#pragma unroll 4
  for (int p = 0; p < pieces; ++p) {
    const float m = ml[p * ml_step];
    M = fmaxf(M, ml[p * ml_step + kBlock] != 0.f ? m : -INFINITY);
  }
  if (!planned && row_pieces(a, listed) <= 1) return;   // written already; here, where the count has arrived with the weights
  f32x4 acc[4] = {};
  float l = 0.f;
#pragma unroll 4
  for (int p = 0; p < pieces; ++p) {
    const float lp = ml[p * ml_step + kBlock], sc = __builtin_amdgcn_exp2f(ml[p * ml_step] - M);
    const bool in = lp != 0.f;   // a piece of weight 0 may hold anything
    l += in ? sc * lp : 0.f;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const f32x4 x = *(const f32x4*)(po + p * o_step + 256 * r4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[r4][e] += in ? sc * x[e] : 0.f;
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int64_t qrow = (int64_t)qb * kBlock + group * 32 + l32;
  if (qrow >= a.lq) return;
  T* const orow = O + a.out_row(qrow) * a.ld + h * kHeadDim + 32 * dt;
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    Tx4 ov;
#pragma unroll
    for (int e = 0; e < 4; ++e) ov[e] = (T)(acc[r4][e] * inv);
    *(Tx4*)(orow + 8 * r4 + 4 * g) = ov;
  }
}

// ------------------------------------------------------------------------------------------------------------
// key lists
// ------------------------------------------------------------------------------------------------------------
// Mask (rows, nk) f32 -> kcnt, kidx (selected ascending, then unselected ascending: argSort(!sel) of
// SparseAttention.swift:175-177 with a stable order). One wave per row.
__global__ __launch_bounds__(256) void lists_from_mask_kernel(const float* __restrict__ mask, int rows, int nk,
                                                              int32_t* __restrict__ kidx,
                                                              int32_t* __restrict__ kcnt) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const float* mrow = mask + (int64_t)row * nk;
  int32_t* krow = kidx + (int64_t)row * nk;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int n_sel = 0;
  for (int j0 = 0; j0 < nk; j0 += 64) {
    const int j = j0 + lane;
    const bool s = j < nk && mrow[j] > 0.5f;
    const uint64_t b = __ballot(s);
    if (s) krow[n_sel + __popcll(b & lt)] = j;
    n_sel += __popcll(b);
  }
  int n_un = n_sel;
  for (int j0 = 0; j0 < nk; j0 += 64) {
    const int j = j0 + lane;
    const bool u = j < nk && !(mrow[j] > 0.5f);
    const uint64_t b = __ballot(u);
    if (u) krow[n_un + __popcll(b & lt)] = j;
    n_un += __popcll(b);
  }
  if (lane == 0) kcnt[row] = n_sel;
}

// Caller-supplied lists as the set they name: the distinct listed blocks inside [0, nk), ascending (kidx_out rows of
// nk entries, kcnt_out). The dense fallback takes lists so: its mask holds a block once, whatever the order, the
// repeats and the indices outside the key range of the list. One wave per row; the set is a bitmap in LDS.
constexpr int kSetWords = 2048;   // 65,536 blocks: K/V buffers and ring layers are below 2 GiB, so nk < 2^16
__global__ __launch_bounds__(64) void set_lists_kernel(const int32_t* __restrict__ kidx,
                                                       const int32_t* __restrict__ kcnt, int nk_stride, int nk,
                                                       int32_t* __restrict__ kidx_out,
                                                       int32_t* __restrict__ kcnt_out) {
  __shared__ unsigned bits[kSetWords];
  const int row = blockIdx.x, lane = threadIdx.x;
  const int words = (nk + 31) / 32;
  for (int w = lane; w < words; w += 64) bits[w] = 0u;
  __syncthreads();
  const int c = min(kcnt[row], nk_stride);
  for (int i = lane; i < c; i += 64) {
    const int j = kidx[(int64_t)row * nk_stride + i];
    if ((unsigned)j < (unsigned)nk) atomicOr(&bits[j >> 5], 1u << (j & 31));
  }
  __syncthreads();
  int32_t* const out = kidx_out + (int64_t)row * nk;
  int base = 0;
  for (int w0 = 0; w0 < words; w0 += 64) {
    unsigned m = w0 + lane < words ? bits[w0 + lane] : 0u;
    const unsigned n = __popc(m), incl = wave_incl_scan(n);
    for (int at = base + (int)(incl - n); m != 0u; m &= m - 1u) out[at++] = 32 * (w0 + lane) + __ffs(m) - 1;
    base += (int)__shfl(incl, 63);
  }
  if (lane == 0) kcnt_out[row] = base;
}

// ------------------------------------------------------------------------------------------------------------
// launch
// ------------------------------------------------------------------------------------------------------------
// compute units of the current device (cached per device)
static int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

// query groups per wave of the bf16 walk: 1 (4 waves of 32 queries, two waves per SIMD) unless FVSR_ATTN_QG=2
// (2 waves of 64 queries, one wave per SIMD)
static int attn_query_groups() {
  static const int qg = [] {
    const char* e = getenv("FVSR_ATTN_QG");
    return (e && e[0] == '2') ? 2 : 1;
  }();
  return qg;
}

// How a call's rows are split. Few rows leave workgroup slots idle and make each row's key list one serial chain, so their
// lists are split into pieces; a piece costs 65 KB of partial result written and read again, and the merge a launch. Measured (12
// heads, us a call with its merge; whole rows, the rows halved .. in equal pieces, pieces of one length):
//   bf16, up to half a row per CU: one workgroup per CU already runs at 70 % of what two reach together, so one item per CU,
//   for every 4 blocks held at most, in equal pieces: planning costs about a microsecond and gains nothing there (48 rows x 16
//   of 16 blocks 31.4, 21.3, 23.0; 72 x 19 of 24 42.3, 26.4, 28.1; 108 x 9 of 19 31.3, 25.6, 26.9). A row of one block
//   stays whole (108 rows x 1 of 27 16.4 with an empty piece to merge, 11.8).
//   bf16, up to a row per CU: two items per CU where lists are long, in pieces of one length of at least 8 blocks (192 rows x
//   32 of 64 78.8, 72.7, 67.9); short lists stay whole (216 x 16 of 18 37.3, 44.4). Two items on a CU take 1.8 times as long
//   a block as one, and the partial results and their merge as long as 5 or 6 blocks, so pieces pay only where they cut the
//   longest list past that, and split_item keeps the rows whole where they don't (all in pieces, now: lists of one length, 240
//   rows x 10 of 60 40.1, 32.8; 192 x 16 of 64 45.2, 41.1; 132 x 30 of 60, in pieces still, 52.4, 52.0 and whole 63.7; lists
//   of about 29 of 48, 192 rows, in pieces still, 65.8, 65.9 and whole 80.9).
//   fp32, where a block costs five times as much: every slot is filled, pieces of one length, down to a block (48 x 16 of 16
//   157, 53, 55; 72 x 19 of 24 212, 92, 77; 108 x 9 of 19 153, 79, 69; 192 x 29 of 48 340, 301, 272; 192 x 32 of 64 423, 356,
//   300).
struct SplitRule {
  int pieces;              // equal pieces of every row (1: whole rows)
  int items, min_blocks;   // or, if items > 0, pieces of one length (split_item)
  int slow, cost;          // unless the longest list is at most slow / 16 pieces + cost blocks long
};
static SplitRule split_rule(int dtype, int64_t rows, int nk, int cus, int64_t max_items) {
  const int64_t one = std::min<int64_t>(cus, max_items), two = std::min<int64_t>(2 * cus, max_items);
  if (rows > kMaxSplitRows) return SplitRule{1};
  if (dtype != FVSR_DTYPE_BF16) return 2 * rows <= two && nk >= 2 ? SplitRule{1, (int)two, 1} : SplitRule{1};
  if (2 * rows <= one && nk >= 8)
    return SplitRule{(int)std::min<int64_t>(std::min<int64_t>(one / rows, nk / 4), kMaxPieces)};
  if (2 * rows <= two && nk >= 48) return SplitRule{1, (int)two, 8, 29, 5};
  return SplitRule{1};
}

// the most items that attentions over up to `rows` rows and nk key blocks split into
int64_t attn_partial_items(int64_t rows, int nk) {
  return std::min<int64_t>(kMaxSplitItems, rows * std::min(kMaxPieces, std::max(1, nk)));
}

int launch_attention(int dtype, AttnArgs a, hipStream_t stream) {
  const int rows = a.heads * a.nq;
  if (rows <= 0) return FVSR_OK;
  const bool half = dtype == FVSR_DTYPE_BF16;
  // two workgroups are resident per CU (64 KB of LDS each in the bf16 walk, 48 in the fp32 one; two waves per SIMD)
  const int slots = std::min(2 * device_cus(), kMaxPersistentWgs);
  const SplitRule rule = a.order ? split_rule(dtype, rows, a.nk, device_cus(), a.part_items) : SplitRule{1};
  a.pieces = rule.pieces;
  a.split_items = rule.items;
  a.split_min = rule.min_blocks;
  a.split_slow = rule.slow;
  a.split_cost = rule.cost;
  a.part_ml = a.part_o + a.part_items * kBlock * kHeadDim;
  const bool direct = rows * a.pieces <= slots || !a.order;   // a workgroup per item
  const dim3 grid(a.split_items > 0 ? a.split_items : direct ? rows * a.pieces : slots);
  if (!direct)
    hipLaunchKernelGGL(attn_order_kernel, dim3(1), dim3(1024), 0, stream, a.kcnt, rows, a.nk_stride, slots, a.order,
                       a.counter);
  auto walk = [&](auto direct_c) {
    constexpr bool DIRECT = decltype(direct_c)::value;
    if (!half)
      hipLaunchKernelGGL(attn_f32_kernel<DIRECT>, grid, dim3(256), 0, stream, a, a.kidx, a.kcnt, (const float*)a.q,
                         (float*)a.o, a.order, a.counter);
    else if (attn_query_groups() == 2)
      hipLaunchKernelGGL((attn_bf16_kernel<2, DIRECT>), grid, dim3(128), 0, stream, a, a.kidx, a.kcnt,
                         (const bf16*)a.q, (bf16*)a.o, a.order, a.counter);
    else
      hipLaunchKernelGGL((attn_bf16_kernel<1, DIRECT>), grid, dim3(256), 0, stream, a, a.kidx, a.kcnt,
                         (const bf16*)a.q, (bf16*)a.o, a.order, a.counter);
  };
  if (direct) walk(std::true_type{});
  else walk(std::false_type{});
  FVSR_HIP_CHECK(hipGetLastError());
  if (a.split_items > 0 || a.pieces > 1) {
    if (half)
      hipLaunchKernelGGL(attn_merge_kernel<bf16>, dim3(4 * rows), dim3(256), 0, stream, a, a.order, (bf16*)a.o);
    else
      hipLaunchKernelGGL(attn_merge_kernel<float>, dim3(4 * rows), dim3(256), 0, stream, a, a.order, (float*)a.o);
    FVSR_HIP_CHECK(hipGetLastError());
  }
  return FVSR_OK;
}

// ------------------------------------------------------------------------------------------------------------
// allocation-free scratch of fvsr_lcsa_attention_noalloc
// ------------------------------------------------------------------------------------------------------------
// The persistent walk's row order (one int32 per (head, query block) row), its work counter and the partial results of
// split rows live in a file-scope device array instead of the context workspace: bytes [0, 256) hold the counter, the
// order starts at byte 256, the partial results follow.
// Every GPU holds its own copy for the life of the process. In host code `scratch` names a host-side stand-in, so
// the device address is taken once per device with hipGetSymbolAddress (noalloc_scratch_init, called by
// fvsr_ctx_create with the device current) and only that address reaches kernels. The order kernel rewrites the
// counter and every order entry it uses on each call, so nothing needs clearing; calls that overlap on one GPU
// share the array and race.
constexpr int kNoAllocRows = 1 << 18;
constexpr size_t kNoAllocOrderBytes = 256 + (size_t)kNoAllocRows * sizeof(int32_t);
constexpr size_t kNoAllocScratchBytes =
    kNoAllocOrderBytes + (size_t)kMaxSplitItems * kPartialFloats * sizeof(float);
static __device__ __align__(256) char scratch[kNoAllocScratchBytes];

static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices] = {};

int noalloc_max_rows() { return kNoAllocRows; }

int noalloc_scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices)
    return set_error(FVSR_ERR_UNSUPPORTED, "device index beyond " + std::to_string(kMaxDevices));
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[device]) return FVSR_OK;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || p == nullptr)
    return set_error(FVSR_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch_ptr[device] = p;
  return FVSR_OK;
}

// `device`'s scratch as the order, counter and partial results of an attention (FVSR_ERR_STATE before
// noalloc_scratch_init). Beyond kNoAllocRows rows the order does not fit: the bf16 walk, whose row order balances it,
// refuses them; the fp32 one runs a workgroup per row.
int noalloc_scratch(int device, int dtype, AttnArgs& a) {
  const int64_t rows = (int64_t)a.heads * a.nq;
  if (rows > kNoAllocRows && dtype == FVSR_DTYPE_BF16)
    return set_error(FVSR_ERR_UNSUPPORTED, "fvsr_lcsa_attention_noalloc: " + std::to_string(rows) +
                                               " (head, query block) rows exceed its static scratch of " +
                                               std::to_string(kNoAllocRows));
  void* p = nullptr;
  if (device >= 0 && device < kMaxDevices) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    p = g_scratch_ptr[device];
  }
  if (!p) return set_error(FVSR_ERR_STATE, "no scratch address for this device: create its context first");
  a.counter = (int32_t*)p;
  a.order = rows <= kNoAllocRows ? (int32_t*)((char*)p + 256) : nullptr;
  a.part_o = (float*)((char*)p + kNoAllocOrderBytes);
  a.part_items = attn_partial_items(rows, a.nk);
  return FVSR_OK;
}

int launch_lists_from_mask(const float* mask, int rows, int nk, int32_t* kidx, int32_t* kcnt, hipStream_t stream) {
  if (rows <= 0) return FVSR_OK;
  hipLaunchKernelGGL(lists_from_mask_kernel, dim3((rows + 3) / 4), dim3(256), 0, stream, mask, rows, nk, kidx, kcnt);
  FVSR_HIP_CHECK(hipGetLastError());
  return FVSR_OK;
}

int launch_set_lists(const int32_t* kidx, const int32_t* kcnt, int rows, int nk_stride, int nk, int32_t* kidx_out,
                     int32_t* kcnt_out, hipStream_t stream) {
  if (rows <= 0) return FVSR_OK;
  if (nk > 32 * kSetWords) return set_error(FVSR_ERR_UNSUPPORTED, "more than 65,536 key blocks");
  hipLaunchKernelGGL(set_lists_kernel, dim3(rows), dim3(64), 0, stream, kidx, kcnt, nk_stride, nk, kidx_out, kcnt_out);
  FVSR_HIP_CHECK(hipGetLastError());
  return FVSR_OK;
}

}  // namespace fvsr
