// fms_inbatch_split.hip -- InBatch() MaxSim with the feature dimension split
// into K slices, for query tiles that do not fit in registers: 16-bit
// features of any dim that is a multiple of 8 other than 32, 64, 96, 128
// (those run the register-resident kernel of fms_inbatch.hip), and fp32
// features of any dim that is a multiple of 4.
//
// S[j, i] = sum_t max_u <Q_i[t], D_j[u]> (forward_layouts.jl:202-225, where
// the reference materialises D'Q chunks and runs an argmax-accumulate); the
// same fused scores and argmax tape as the other in-batch kernel.
//
// A plan lists the call's document chunks that hold a valid row, in document
// order (a document without one keeps one chunk, all masked, so that it
// closes), and cuts the list into R ranges of equal length at document
// boundaries.  Work item = one range x kRows query rows (a query row is a
// 32-token tile of a query: query v / ntq, tokens 32 (v % ntq) ..; of all queries'
// tokens as one run where that leaves fewer tiles, kFlat).  Blocks of 4
// waves, one per CU for 16-bit features and two for fp32, each walk their
// items in turn (a persistent grid).  An item's chunks are taken kCg at a time
// whatever documents they belong to (a chunk group: 6 chunks for 16-bit
// features, 3 for fp32); per group the block runs the whole K loop:
//   * K advances by a slice of 128 bytes of every row (64 features of a
//     16-bit type, 32 of fp32).  The chunks' slice (shared by the four
//     waves) goes HBM/L2 -> LDS with direct buffer-to-LDS loads of whole rows
//     (layout below).  A wave's own query rows' fragments are loaded straight
//     into registers.  Rows past the document or the query, and units past the
//     row (the last slice of a dim that is not a multiple of it) read zeros
//     (buffer bounds);
//   * the block's slices (items, their groups, their K slices, in order)
//     form one stream with three stages: slice task p + 2 is requested
//     while task p is multiplied, across group and item boundaries, so an
//     item's first slices arrive while the previous item folds and closes;
//     one barrier per task (every wave's share of task p + 1 has landed, and
//     every wave is done with the stage of task p, which the request of task
//     p + 3 then refills).  It stands before the last quarter of task p's
//     MFMAs, and task p + 1's first fragments are read behind it, so neither
//     the barrier nor the LDS latency holds up the matrix cores;
//   * wave w holds the accumulators of query rows 2w, 2w + 1 for the whole
//     chunk group (2 x kCg 32x32 tiles): each query fragment read feeds kCg
//     MFMA chains and each document fragment read two;
//   * 16-bit: one v_mfma_f32_32x32x16 per unit pair.  fp32: the 16 bytes of
//     a unit pair are four k-blocks of v_mfma_f32_32x32x2f32; dword e of
//     the lanes of half h is feature 8m + 4h + e of the slice, the same
//     bijection for both operands, so the four MFMAs sum the 8 features of
//     the unit pair;
//   * after a group's last slice each accumulator tile is folded, chunk by
//     chunk in list order, into the running max / argmax exactly as the
//     scans fold (first valid row taken, then strictly greater), and a
//     document's last chunk closes it: wave halves merged, tape rows and the
//     score written straight to global memory.  Without a tape (args null) the
//     fold is the max3 tree alone.
// Item -> (range, query group) is XCD-aware: an XCD's 32 CUs hold a few query
// groups x several ranges at a time: a chunk is read by the CUs of several query
// groups and a query row by those of several ranges (split_slot, split_cut).
//
// Measured, us per call on documents of U[Td / 3, Td] tokens, scores alone / with
// the tape, against one document per item, all its chunks multiplied and a
// task's loads ahead of its MFMAs: bf16, d = 768, 256 x 256, Td = 180: 655 / 656 ->
// 408 / 451 (0.96 PFLOP/s on valid tokens); 512 x 512 2591 / 2605 -> 1532 / 1710;
// fp16, d = 256, 512 x 512, Td = 300 1980 / 1990 -> 1019 / 1260; fp32, d = 128, 512 x
// 512 3289 / 3308 -> 2116 / 2209; 64 x 64 bf16, d = 768 47 -> 45.  Full documents: bf16
// 256 x 256 663 -> 543.  Bound by the MFMAs and, in 16 bits, by the one wave per
// SIMD that the accumulators leave: its fold and close run with the matrix cores
// idle.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "fms_device.hpp"
#include "fms_group.hpp"
#include "fms_inbatch_split.hpp"
#include "fms_scan.hpp"

namespace fms {

namespace {

constexpr int kSpWaves = 4;
constexpr int kRows = 2 * kSpWaves;     // query rows per block (two per wave)
constexpr int kSliceBytes = 128;        // bytes of every row per K step
constexpr int kPairs = kSliceBytes / 32;  // unit pairs per slice (4)
constexpr int kStages = 3;              // document slice stages in LDS (2 slices ahead)
static_assert(kTile == 8 * kSpWaves, "every wave copies 8 whole rows of each chunk");
constexpr int kQLoads = 2 * kPairs;     // query fragment loads per slice and wave

// The chunk group per element size.  kCg document chunks per group, kBlocks
// blocks per CU.  16-bit: six chunks, one block (a wave holds 12 accumulator
// tiles and its query fragments in about 424 registers).  fp32: three
// chunks, two blocks (256 registers): its MFMAs take 8 times as long per
// byte, so a second wave per SIMD covers the first one's per-slice work
// (measured at the C3 shape: 3.55 -> 3.39 ms), while for 16-bit features the
// halved reuse of each query fragment costs more than that (2.85 -> 3.71 ms).
template <int kEsz>
struct SplitShape {
  static constexpr int kCg = kEsz == 4 ? 3 : 6;
  static constexpr int kBlocks = kEsz == 4 ? 2 : 1;
  static constexpr int kDFrags = kCg * kPairs;  // 1 KB blocks of a document slice
  // Vector memory operations per slice and wave: kCg document copies into
  // LDS, then the query fragment loads into registers.
  static constexpr int kOpsPerSlice = kCg + kQLoads;
  // Issued after a slice's document copies by the time that slice is read:
  // its own query loads and the two slices requested since.
  static constexpr int kAfterCopies = kQLoads + (kStages - 2) * kOpsPerSlice;
  static_assert(kAfterCopies < 64, "vmcnt field");
};
constexpr int kMaxCg = SplitShape<2>::kCg;  // the largest group (range checks)
static_assert(SplitShape<4>::kCg <= kMaxCg, "range checks cover every shape");
constexpr int kSpXcds = 8;

// The block's waves have all landed their loads of the slice to be read next
// (each leaves only its kVm most recent loads in flight) and finished their
// LDS accesses; the asm statements keep the compiler from moving LDS
// accesses across.
template <int kVm>
__device__ __forceinline__ void slice_barrier() {
  static_assert(kVm >= 0 && kVm < 64, "vmcnt field");
  asm volatile("" ::: "memory");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kVm) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// acc += the products of one unit pair (16 bytes per lane of each operand):
// kMmaPerPair MFMAs.
template <class Op>
__device__ __forceinline__ typename Op::Acc mma_pair(u32x4 a, u32x4 b, typename Op::Acc acc) {
  if constexpr (Op::kEsz == 4) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = Op::mma(a[e], b[e], acc);
    return acc;
  } else {
    return Op::mma(a, b, acc);
  }
}

// base[at] = v for at < n (wave-uniform base and n), nothing past it.  The task
// loop's stores go through this, none under a branch on the lane: divergent
// control flow there makes the compiler restructure the whole loop.  (A device
// function: a resource local to a lambda keeps the host compile from emitting
// the kernel's launch stub.)
__device__ __forceinline__ void store_below(const void* base, int n, int at, uint32_t v) {
  __builtin_amdgcn_raw_buffer_store_b32(v, make_rsrc_u(base, (uint32_t)n * 4u), at * 4, 0, 0);
}

// A wave's 16 bytes per lane HBM/L2 -> LDS, and into registers, with a scalar
// offset (device functions, not lambdas, for the same reason).
__device__ __forceinline__ void copy16_lds(rsrc_t r, u32x4* dst, int voff, int soff) {
  typedef __attribute__((address_space(3))) void* lds_void_t;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t)dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ u32x4 load16_at(rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// Valid-row words of the call, one launch before the scan: plan[j * nch + c]
// bit r = row 32c + r of document j is below Td and unmasked; plan[ndw + v]
// bit r = token 32 (v % ntq) + r of query v / ntq is below Tq and unmasked.
// The scan reads them with scalar loads (a wave-uniform word per chunk or
// query row), which leaves the vector-memory counter to the slice stream.
__global__ void __launch_bounds__(256) split_plan_kernel(const uint8_t* dm, const uint8_t* qm,
                                                         int Bd, int Td, int nch, int Bq, int Tq,
                                                         int ntq, uint32_t* plan) {
  const int64_t ndw = (int64_t)Bd * nch, total = ndw + (int64_t)Bq * ntq;
  const int lane = threadIdx.x & 63;
  // two words per wave and pass: lanes 0..31 word w, lanes 32..63 word w + 1
  for (int64_t w = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 2; w < total;
       w += (int64_t)gridDim.x * 8) {
    const int64_t wi = w + (lane >> 5);
    bool bit = false;
    if (wi < ndw) {
      const int64_t j = wi / nch;
      const int row = (int)(wi - j * nch) * kTile + (lane & 31);
      bit = row < Td && (dm == nullptr || dm[j * Td + row] != 0);
    } else if (wi < total) {
      const int64_t v = wi - ndw, i = v / ntq;
      const int t = (int)(v - i * ntq) * kTile + (lane & 31);
      bit = t < Tq && (qm == nullptr || qm[i * Tq + t] != 0);
    }
    const uint64_t b = __ballot(bit);
    if ((lane & 31) == 0 && wi < total) plan[wi] = (uint32_t)(b >> (lane & 32));
  }
}

// The chunk list: entry {valid rows, document, chunk | last << 31, 0} per listed
// chunk (see above), and rs[r], the first entry of range r (rs[R]: the entries'
// number).  byDocs: range r starts at document r Bd / R; otherwise at the first
// document whose first entry is at or past r / R of the list.
//
// A block lists kListThreads documents, a thread per document.  With several
// blocks split_count_kernel has left each one's number of entries in counts, and
// every block adds up those before it and all of them; one block counts for itself.
// (All documents by one block, kListThreads at a time, were a serial stretch ahead of
// the scan.  us per call of 8 queries of 32 tokens, one block / a block per 1024: d = 40,
// fp16, 5000 documents of 60 .. 180 tokens 121 / 99, with the tape 155 / 137; d = 256, bf16,
// 50000 of them 1622 / 1318; d = 8, 200000 documents of one chunk 1523 / 1004; 2100 63 / 56.)
constexpr int kListThreads = 1024;

// f(chunk, valid rows) for the chunks of document j with a valid row.
template <class F>
__device__ __forceinline__ void each_chunk(const uint32_t* plan, int nch, int64_t j, F f) {
  constexpr int kWords = 8;  // plan words in flight per thread
  const uint32_t* const words = plan + j * nch;
  for (int c0 = 0; c0 < nch; c0 += kWords) {
    uint32_t m[kWords];
#pragma unroll
    for (int i = 0; i < kWords; ++i) m[i] = c0 + i < nch ? words[c0 + i] : 0u;
#pragma unroll
    for (int i = 0; i < kWords; ++i)
      if (m[i] != 0u) f(c0 + i, m[i]);
  }
}

// Entries of document j (0 past the last document).
__device__ __forceinline__ int doc_entries(const uint32_t* plan, int nch, int64_t j, int Bd) {
  if (j >= Bd) return 0;
  int n = 0;
  each_chunk(plan, nch, j, [&](int, uint32_t) { ++n; });
  return n > 0 ? n : 1;
}

// Exclusive prefix of v over the block and its total (two barriers).
__device__ __forceinline__ int list_scan(int v, int& total) {
  __shared__ int wsum[kListThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  int before = x - v;
  total = 0;
#pragma unroll
  for (int i = 0; i < kListThreads / 64; ++i) {
    if (i < w) before += wsum[i];
    total += wsum[i];
  }
  __syncthreads();
  return before;
}

__global__ void __launch_bounds__(kListThreads) split_count_kernel(const uint32_t* plan, int Bd, int nch,
                                                                   int32_t* counts) {
  int total;
  list_scan(doc_entries(plan, nch, (int64_t)blockIdx.x * kListThreads + threadIdx.x, Bd), total);
  if (threadIdx.x == 0) counts[blockIdx.x] = total;
}

__global__ void __launch_bounds__(kListThreads) split_list_kernel(const uint32_t* plan, int Bd, int nch,
                                                                  int R, int byDocs, const int32_t* counts,
                                                                  uint4* list, int32_t* rs) {
  int base = 0, all = 0;
  if (gridDim.x > 1) {
    int mine = 0, every = 0;
    for (int b = threadIdx.x; b < (int)gridDim.x; b += kListThreads) {
      const int c = counts[b];
      every += c;
      mine += b < (int)blockIdx.x ? c : 0;
    }
    list_scan(mine, base);
    list_scan(every, all);
  }
  const int64_t jt = (int64_t)blockIdx.x * kListThreads + threadIdx.x;
  const int n = doc_entries(plan, nch, jt, Bd);
  int total;
  const int e0 = base + list_scan(n, total);
  if (gridDim.x == 1) all = total;
  if (n == 0) return;
  const int j = (int)jt;
  // the range that document j, first entry e, belongs to
  auto range_of = [&](int j, int e) {
    return byDocs ? (int)(((int64_t)j * R + R - 1) / Bd) : (int)(((int64_t)e * R) / all);
  };
  int e = e0;
  each_chunk(plan, nch, j, [&](int c, uint32_t m) {
    list[e] = make_uint4(m, (uint32_t)j, (uint32_t)c | ((e + 1 == e0 + n) ? 0x80000000u : 0u), 0u);
    ++e;
  });
  if (e == e0) list[e] = make_uint4(0u, (uint32_t)j, 0x80000000u, 0u);
  // the ranges that start at the next document (or, past the last one, at the end)
  const int en = e0 + n, lo = range_of(j, e0), hi = j + 1 == Bd ? R : range_of(j + 1, en);
  if (j == 0) rs[0] = 0;
  for (int r = lo + 1; r <= hi; ++r) rs[r] = en;
}

// Slot x of the block order -> (range, query group); qg = nqg marks a slot with
// no work.  Slots are dealt round-robin to the 8 XCDs (slot x runs on XCD x % 8:
// the grid is a multiple of 8 and each block walks slots blockIdx.x + n *
// gridDim.x).  XCD x takes every xq-th query group and every (8 / xq)-th range,
// and goes through its ranges for one query group before the next.
__device__ __forceinline__ int split_slot(int x, int nqg, int R, int xq, int& qg) {
  const int xcd = x % kSpXcds, k = x / kSpXcds, xr = kSpXcds / xq;
  const int nrx = (R + xr - 1) / xr;
  const int r = (k % nrx) * xr + xcd / xq;
  const int g = (k / nrx) * xq + xcd % xq;
  qg = r < R && g < nqg ? g : nqg;
  return r;
}

// kWhole: rows are whole slices (rowbytes a multiple of kSliceBytes, as at
// d = 768 in 16 bits or d = 128 in fp32), so no unit lies past a row's end
// and the slice's byte offset goes to the loads' scalar offset.
// kFlat: the queries' tokens are one run of A.Tq = Bq * qtok tokens (A.Bq = 1), cut
// into tiles whatever query they belong to, so short queries (and the last tile of
// long ones) multiply no padding; a close stores each token's maximum (A.St), and
// split_token_sum_kernel sums the queries.  The launcher says when.  us per call
// against a query per tile, scores alone / with the tape, documents of Td / 3 .. Td
// tokens: bf16, d = 256, 512 x 512, Td = 300: 978 / 1179 -> 314 / 379 at 9 query tokens,
// 659 / 826 at 20, and 40 tokens (two tiles) about 1960 / 2360 -> 1225 / 1502; bf16,
// d = 768, 200 x 200, Td = 180: 289 / 316 -> 112 / 122 at 9, 177 / 195 at 16; fp32, d = 128,
// 200 x 200: 386 / 401 -> 174 / 184 at 9, 278 / 292 at 20.
template <class Op, bool kWhole, bool kTape, bool kFlat>
__global__ void __launch_bounds__(64 * kSpWaves, SplitShape<Op::kEsz>::kBlocks)
    inbatch_split(const InBatchSplitArgs A) {
  typedef typename Op::Acc Acc;
  typedef SplitShape<Op::kEsz> Shape;
  constexpr int kCg = Shape::kCg, kDFrags = Shape::kDFrags, kAfterCopies = Shape::kAfterCopies;
  // three arrays, not one indexed by stage: the compiler then sees that a copy
  // into one stage cannot alias reads of another
  __shared__ u32x4 dbuf0[kDFrags * 64], dbuf1[kDFrags * 64], dbuf2[kDFrags * 64];
  static_assert(kStages == 3, "three stages, and the task loop below is unrolled by three");

  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int r32 = lane & 31, h = lane >> 5;

  const int rowbytes = A.rowbytes, Tq = A.Tq, Td = A.Td, ntq = A.ntq, Bd = A.Bd, nqg = A.nqg, R = A.R, xq = A.xq;
  const int nslices = (rowbytes + kSliceBytes - 1) / kSliceBytes;
  const int nqv = A.Bq * ntq;
  const int G = gridDim.x;
  // The plan is read through the constant address space: scalar loads
  // (wave-uniform words, lgkmcnt), nothing in the vector-memory count that the
  // slice waits rely on.  The kernel never writes it.
  typedef __attribute__((address_space(4))) const uint32_t* cword_ptr;
  typedef __attribute__((address_space(4))) const int32_t* cint_ptr;
  const cword_ptr clist = (cword_ptr)(uintptr_t)A.list;
  const cint_ptr crs = (cint_ptr)(uintptr_t)A.rs;
  const cword_ptr qmask = (cword_ptr)(uintptr_t)A.qwords;

  // This block's slots with work, in order: the first at or after x.
  auto next_slot = [&](int x) {
    for (; x < A.nslots; x += G) {
      int qg;
      const int r = split_slot(x, nqg, R, xq, qg);
      if (qg < nqg && crs[r] < crs[r + 1]) break;
    }
    return x;
  };

  // Query rows of a wave for query group qg: query, first token, token count.
  struct Rows {
    int qv[2], qi[2], qt0[2], qtn[2];
    int tq0[2];  // kFlat tape: the first token's query
  };
  auto rows_of = [&](int qg) {
    Rows Rw;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int v = qg * kRows + 2 * wave + q;
      const bool live = v < nqv;
      Rw.qv[q] = live ? v : -1;
      Rw.qi[q] = live ? v / ntq : 0;
      Rw.qt0[q] = live ? (v - Rw.qi[q] * ntq) * kTile : 0;
      Rw.qtn[q] = live ? std::min(kTile, Tq - Rw.qt0[q]) : 0;
      if constexpr (kFlat && kTape) Rw.tq0[q] = Rw.qt0[q] / A.qtok;
    }
    return Rw;
  };

  // ---- the load stream ---------------------------------------------------------
  // Per task and wave: kCg document copies into LDS (the four waves together
  // copy the whole slice), then this wave's own query fragments (2 rows x
  // kPairs unit pairs) into registers, lane l reading row l % 32, unit 2m +
  // l / 32 of the slice.  Each chunk of the group has a buffer resource of its
  // own (its rows up to the document's end; empty past the item's last chunk
  // and past the block's last task: the same operations, no memory traffic), so
  // a lane's offset is the same for every chunk, group and slice.
  // Document copies read whole rows: a wave's copy of a chunk is its rows
  // 8w .. 8w + 7 (1 KB, 8 cache lines), lane l taking row 8w + l / 8 and the
  // unit that leaves the chunk row-major with each row's 8 units
  // XOR-swizzled: unit u of row r at r * 8 + (u ^ key(r)), key(r) =
  // (r / 2) % 8.  The fragment reads (lane: row r32, unit 2m + h) then fall
  // on 16 distinct 16-byte bank groups for any 16 consecutive lanes.
  const int crow = 8 * wave + (lane >> 3);
  const int copy_off = ((lane & 7) ^ ((crow >> 1) & 7)) * 16;
  const int dvoff = crow * rowbytes, qvoff = r32 * rowbytes + h * 16;
  int roff[kPairs];  // fragment m of a chunk: u32x4 index in the chunk's 4 KB
#pragma unroll
  for (int m = 0; m < kPairs; ++m) roff[m] = r32 * 8 + ((2 * m + h) ^ ((r32 >> 1) & 7));
  int is_slot = next_slot(blockIdx.x), is_e = 0, is_end = 0, is_s = 0;
  rsrc_t rdoc[kCg], rq[2];
  auto set_issue_group = [&]() {
#pragma unroll
    for (int c = 0; c < kCg; ++c) {
      const bool in = is_e + c < is_end;
      const int64_t e = in ? is_e + c : 0;
      const int j = (int)clist[e * 4 + 1], ch = (int)(clist[e * 4 + 2] & 0x7fffffffu);
      const int rows = in ? std::min(kTile, Td - ch * kTile) : 0;
      rdoc[c] = make_rsrc_u(A.D + ((int64_t)j * Td + ch * kTile) * rowbytes,
                            rows > 0 ? (uint32_t)rows * (uint32_t)rowbytes : 0u);
    }
  };
  auto set_issue_item = [&]() {
    if (is_slot < A.nslots) {
      int qg;
      const int r = split_slot(is_slot, nqg, R, xq, qg);
      is_e = crs[r];
      is_end = crs[r + 1];
      const Rows Rw = rows_of(qg);
#pragma unroll
      for (int q = 0; q < 2; ++q)
        rq[q] = make_rsrc_u(A.Q + ((int64_t)Rw.qi[q] * Tq + Rw.qt0[q]) * rowbytes,
                            (uint32_t)Rw.qtn[q] * (uint32_t)rowbytes);
    } else {
      is_e = is_end = 0;
      rq[0] = rq[1] = make_rsrc_u(A.Q, 0u);
    }
    set_issue_group();
  };
  set_issue_item();
  // Query fragments of kStages tasks in flight: set k holds tasks 3n + k.
  u32x4 qf[kStages][2][kPairs];
  // Load i of a task (0 .. kOpsPerSlice - 1): a document copy or a query fragment.
  auto issue_one = [&](auto SETc, auto Ic) {
    constexpr int kSet = decltype(SETc)::value, i = decltype(Ic)::value;
    u32x4* const dst = kSet == 0 ? dbuf0 : kSet == 1 ? dbuf1 : dbuf2;
    const int s0 = is_s * kSliceBytes;  // uniform: the loads' scalar offset
    if constexpr (i < kCg) {
      if constexpr (kWhole) {
        copy16_lds(rdoc[i], &dst[i * 256 + wave * 64], dvoff + copy_off, s0);
      } else {
        // A unit past the row end is pushed out of range with all low 31 bits set
        // (branch-free: a select here became divergent branches around the loads).
        const int past = -(int)(s0 + copy_off >= rowbytes) & 0x7fffffff;
        copy16_lds(rdoc[i], &dst[i * 256 + wave * 64], (dvoff + s0 + copy_off) | past, 0);
      }
    } else {
      constexpr int q = (i - kCg) / kPairs, m = (i - kCg) % kPairs;
      if constexpr (kWhole) {
        qf[kSet][q][m] = load16_at(rq[q], qvoff + m * 32, s0);
      } else {
        const int past = -(int)(s0 + (2 * m + h) * 16 >= rowbytes) & 0x7fffffff;
        qf[kSet][q][m] = load16_at(rq[q], (qvoff + s0 + m * 32) | past, 0);
      }
    }
  };
  auto advance = [&]() {
    if (++is_s < nslices) return;
    is_s = 0;
    is_e += kCg;
    if (is_e < is_end) {
      set_issue_group();
    } else {
      is_slot = next_slot(is_slot + G);
      set_issue_item();
    }
  };

  // ---- the compute side -----------------------------------------------------------
  int c_slot = next_slot(blockIdx.x), c_e = 0, c_end = 0, c_s = 0;
  Rows Rw{};
  auto set_compute_item = [&]() {
    int qg = 0;
    c_e = c_end = 0;
    if (c_slot < A.nslots) {
      const int r = split_slot(c_slot, nqg, R, xq, qg);
      c_e = crs[r];
      c_end = crs[r + 1];
    }
    Rw = rows_of(qg);
  };
  set_compute_item();
  if (c_slot >= A.nslots) return;
  int64_t ntasks = 0;  // (items x groups x slices can pass 2^31 at extreme shapes)
  for (int x = c_slot; x < A.nslots; x = next_slot(x + G)) {
    int qg;
    const int r = split_slot(x, nqg, R, xq, qg);
    ntasks += (int64_t)((crs[r + 1] - crs[r] + kCg - 1) / kCg) * nslices;
  }

  // Running max of both rows.  With a tape: (max, slot) as the scans keep them.
  // Without: the max alone, the score of the document's first valid row (which
  // stands when it is NaN, see take_first_row) and whether there was one.
  float mx[2] = {-INFINITY, -INFINITY}, first[2] = {-INFINITY, -INFINITY};
  int slot[2] = {-1, -1};
  bool any = false;

  // Close document j for both query rows: wave halves merged, tape row and
  // score written straight to global memory.  Both rows' running max starts
  // again, a row past the last query (whose folds saw zeros) included.
  auto close_doc = [&](int j) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (Rw.qv[q] >= 0) {
        const uint32_t qw = qmask[Rw.qv[q]];
        const bool tv = ((qw >> r32) & 1u) != 0u;
        const int64_t p = (int64_t)Rw.qi[q] * Bd + j;
        float part;
        if constexpr (kTape) {
          int tok = slot_to_token(slot[q], h);
          float m = mx[q];
          merge_halves(m, tok, h);
          part = (tv && tok != 0) ? m : 0.0f;
          if constexpr (kFlat) {
            // (row / qtok by a 16-bit reciprocal, exact below 2^16 / qtok; computed
            // here, not kept: two more registers a lane made the accumulators move)
            const int row = r32 + (Rw.qt0[q] - Rw.tq0[q] * A.qtok);
            const int i = (int)(((uint32_t)row * A.qrecip) >> 16);
            const int past = -(int)(lane >= Rw.qtn[q]) & 0x1fffffff;
            store_below(A.args + ((int64_t)Rw.tq0[q] * Bd + j) * A.qtok, (kTile + 1) * Bd * A.qtok,
                        (i * (Bd - 1) * A.qtok + row) | past, (uint32_t)(tv ? tok : 0));
          } else
            store_below(A.args + p * Tq + Rw.qt0[q], Rw.qtn[q], lane, (uint32_t)(tv ? tok : 0));
        } else {
          const float m = merge_halves_max(mx[q]);
          const uint32_t nf = is_nan_bits(first[q]) ? 1u : 0u;
          const bool nan_first = (nf | lane_xor32(nf, h)) != 0u;
          part = tv && any ? (nan_first ? __builtin_bit_cast(float, 0x7fc00000u) : m) : 0.0f;
        }
        if constexpr (kFlat) {
          store_below(A.St + ((int64_t)j * ntq * kTile + Rw.qt0[q]), Rw.qtn[q], lane,
                      __builtin_bit_cast(uint32_t, part));
        } else {
          const float score = half_sum(part);
          const float nf = (float)__builtin_popcount(qw);
          const float inv = 1.0f / (nf > 1.0f ? nf : 1.0f);
          const float sc = A.norm && ntq == 1 ? score * inv : score;
          const float* const out = ntq > 1 ? A.St + ((int64_t)Rw.qv[q] * Bd + j) : A.S + p;
          store_below(out, 1, lane, __builtin_bit_cast(uint32_t, sc));
        }
      }
      mx[q] = -INFINITY;
      first[q] = -INFINITY;
      slot[q] = -1;
    }
    any = false;
  };

  // Fold one chunk's scores of query row q (valid rows m32, chunk ch).
  auto fold = [&](float (&s)[16], uint32_t m32, int ch, int q) {
    if constexpr (kTape) {
      take_first_row(s, m32, h, ch, mx[q], slot[q]);
      if (m32 == 0xffffffffu) fold_tree<true>(s, ch * 16, mx[q], slot[q]);
      else update_chunk(s, m32, h, ch, mx[q], slot[q]);
    } else {
      if (!any) {  // (m32 != 0)
        const int row = __builtin_ctz(m32);
        const int reg = ((row >> 3) << 2) | (row & 3);
        f32x16 sv;
#pragma unroll
        for (int r = 0; r < 16; ++r) sv[r] = s[r];
        const float v = sv[reg];
        first[q] = h == ((row >> 2) & 1) ? v : -INFINITY;
      }
      if (m32 != 0xffffffffu) {
        const uint32_t bits = m32 >> (4 * h);
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = ((bits >> acc_row(r, 0)) & 1u) ? s[r] : -INFINITY;
      }
      fold_max(s, mx[q]);
    }
  };

  Acc acc[kCg][2];
  u32x4 a[2][kCg];  // document fragments of two unit pairs
  auto read_pair = [&](auto SETc, int m, int c, u32x4& dst) {
    constexpr int kSet = decltype(SETc)::value;
    const u32x4* const B = kSet == 0 ? dbuf0 : kSet == 1 ? dbuf1 : dbuf2;
    dst = B[c * 256 + roff[m]];
  };

  // Task p.  On entry its slice is in LDS and its pair 0 fragments are in a[0].
  // Pair m's MFMAs run while pair m + 1's fragments are read; task p + 2's loads
  // go out one by one between the first MFMAs; before pair 3's, the wait and
  // barrier for task p + 1's slice (exactly kAfterCopies vector operations were
  // issued after its copies: its own query loads and the whole of task p + 2),
  // then task p + 1's pair 0 fragments are read.  Each unit (a fragment read, a
  // load, the MFMAs of one chunk) is fenced: the compiler otherwise puts every
  // read right before its MFMAs and all loads ahead of them.
  auto step = [&](auto SETc) {
    constexpr int kSet = decltype(SETc)::value;
    typedef std::integral_constant<int, (kSet + 1) % kStages> NextSet;
    typedef std::integral_constant<int, (kSet + 2) % kStages> IssueSet;
    constexpr int kOps = Shape::kOpsPerSlice;
    auto pair_mma = [&](auto Mc, auto FIRSTc) {
      constexpr int m = decltype(Mc)::value;
      constexpr bool kZero = decltype(FIRSTc)::value;
      static_for<0, kCg>([&](auto Cc) {
        constexpr int c = decltype(Cc)::value;
        if constexpr (m + 1 < kPairs) read_pair(SETc, m + 1, c, a[(m + 1) & 1][c]);
        else read_pair(NextSet(), 0, c, a[0][c]);
        // loads of task p + 2: spread over pairs 0 .. kPairs - 2
        constexpr int units = kCg * (kPairs - 1), u = m * kCg + c;
        if constexpr (m < kPairs - 1)
          static_for<u * kOps / units, (u + 1) * kOps / units>(
              [&](auto Ic) { issue_one(IssueSet(), Ic); });
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 2; ++q)
          acc[c][q] = mma_pair<Op>(a[m & 1][c], qf[kSet][q][m], kZero ? Acc{} : acc[c][q]);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    static_assert(kPairs == 4, "pair 3 reads into the fragment set pair 0 used");
    auto multiply = [&](auto FIRSTc) {
      pair_mma(std::integral_constant<int, 0>(), FIRSTc);
      pair_mma(std::integral_constant<int, 1>(), std::false_type());
      pair_mma(std::integral_constant<int, 2>(), std::false_type());
      slice_barrier<kAfterCopies>();
      pair_mma(std::integral_constant<int, 3>(), std::false_type());
    };
    if (c_s == 0) multiply(std::true_type());
    else multiply(std::false_type());
    advance();

    if (++c_s == nslices) {
      c_s = 0;
#pragma unroll
      for (int c = 0; c < kCg; ++c) {
        if (c_e + c >= c_end) continue;
        const int64_t e = c_e + c;
        const uint32_t m32 = clist[e * 4], j = clist[e * 4 + 1], ci = clist[e * 4 + 2];
        if (m32 != 0u) {
          const int ch = (int)(ci & 0x7fffffffu);
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            float s[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = acc[c][q][r];
            fold(s, m32, ch, q);
          }
          any = true;
        }
        if (ci >> 31) close_doc((int)j);
      }
      c_e += kCg;
      if (c_e >= c_end) {
        c_slot = next_slot(c_slot + G);
        set_compute_item();
      }
    }
  };

  // The first two tasks' loads, then the steps (past the block's last task the
  // loads are empty).  The only branches between steps leave the loop: none
  // skips a step.
  auto issue_all = [&](auto SETc) {
    static_for<0, Shape::kOpsPerSlice>([&](auto Ic) {
      issue_one(SETc, Ic);
      __builtin_amdgcn_sched_barrier(0);  // in this order: the waits count them
    });
  };
  issue_all(std::integral_constant<int, 0>());
  advance();
  issue_all(std::integral_constant<int, 1>());
  advance();
  slice_barrier<kAfterCopies>();
#pragma unroll
  for (int c = 0; c < kCg; ++c) read_pair(std::integral_constant<int, 0>(), 0, c, a[0][c]);
  for (int64_t p = 0;;) {
    step(std::integral_constant<int, 0>());
    if (++p == ntasks) break;
    step(std::integral_constant<int, 1>());
    if (++p == ntasks) break;
    step(std::integral_constant<int, 2>());
    if (++p == ntasks) break;
  }
  slice_barrier<0>();  // the empty requests past the last task
}

// S[i, j] = sum over tiles tb (in order) of St[i * ntq + tb, j], times
// 1 / max(valid tokens of query i, 1) when normalising.
__global__ void __launch_bounds__(256) split_tile_sum_kernel(const float* St, int ntq, int Bq,
                                                             int Bd, const uint8_t* qm, int Tq,
                                                             int norm, float* S) {
  __shared__ int cnt;
  for (int i = blockIdx.y; i < Bq; i += gridDim.y) {
    float inv = 1.0f;
    if (norm) {
      if (threadIdx.x == 0) cnt = 0;
      __syncthreads();
      int c = 0;
      for (int t = threadIdx.x; t < Tq; t += 256) c += qm ? (qm[(int64_t)i * Tq + t] != 0) : 1;
      atomicAdd(&cnt, c);
      __syncthreads();
      const float nf = (float)cnt;
      inv = 1.0f / (nf > 1.0f ? nf : 1.0f);
      __syncthreads();
    }
    for (int jj = blockIdx.x * 256 + threadIdx.x; jj < Bd; jj += gridDim.x * 256) {
      float s = 0.0f;
      for (int tb = 0; tb < ntq; ++tb) s += St[((int64_t)i * ntq + tb) * Bd + jj];
      S[(int64_t)i * Bd + jj] = norm ? s * inv : s;
    }
  }
}

// S[i, j] = the sum of query i's token maxima St[j][i * Tq ..] (rows of nr tokens), a
// thread per (i, j), added as half_sum adds a tile's 32 tokens and tile after tile,
// so scores are bit for bit those of a query per tile; normalised as above.
__global__ void __launch_bounds__(256) split_token_sum_kernel(const float* St, int64_t nr, int Bq, int Bd,
                                                              const uint8_t* qm, int Tq, int norm,
                                                              float* S) {
  const int64_t n = (int64_t)Bq * Bd;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    const int64_t j = e / Bq;
    const int i = (int)(e - j * Bq);
    const float* const x = St + j * nr + (int64_t)i * Tq;
    float s = 0.0f;
    for (int t0 = 0; t0 < Tq; t0 += kTile) {
      float row[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float quad[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float v[4];
#pragma unroll
          for (int l = 0; l < 4; ++l) {
            const int t = t0 + 16 * h + 4 * k + l;
            v[l] = t < Tq ? x[t] : 0.0f;
          }
          quad[k] = (v[0] + v[1]) + (v[2] + v[3]);
        }
        row[h] = (quad[0] + quad[3]) + (quad[2] + quad[1]);
      }
      s += row[0] + row[1];
    }
    if (norm) {
      int c = qm ? 0 : Tq;
      if (qm)
        for (int t = 0; t < Tq; ++t) c += qm[(int64_t)i * Tq + t] != 0;
      s *= 1.0f / (float)(c > 1 ? c : 1);
    }
    S[(int64_t)i * Bd + j] = s;
  }
}

}  // namespace

bool inbatch_split_supported(int esz, int64_t dim, int64_t Tq, int64_t Td, int64_t Bq,
                             int64_t Bd, const void* Q, const void* D) {
  const bool al = ((reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(D)) & 15u) == 0;
  const int64_t rowbytes = dim * esz;
  const int64_t ntq = Tq > kTile ? (Tq + kTile - 1) / kTile : 1;
  const int64_t nqg = (Bq * ntq + kRows - 1) / kRows, ndx = (Bd + kSpXcds - 1) / kSpXcds;
  // 32-bit buffer offsets: a chunk's rows, a query tile's rows; 32-bit counts:
  // the chunk list, the slots (ranges are at most as many as documents)
  const int64_t lim = ((int64_t)1 << 31) - 4096;
  return (esz == 2 || esz == 4) && dim > 0 && rowbytes % 16 == 0 && al && Tq >= 1 && Td >= 0 &&
         Bq >= 1 && Bd >= 1 && Bq * ntq <= ((int64_t)1 << 30) && Bd <= ((int64_t)1 << 26) &&
         (Td + kTile * kMaxCg) * rowbytes < lim && kTile * rowbytes < lim &&
         Bd * ((Td + kTile - 1) / kTile + 1) < lim && nqg <= lim / kSpXcds / ndx;
}

namespace {

// Compute units of the current device (cached per device; gfx950: 256).
int device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 256;
  if (dev < 64) {
    const int c = cache[dev].load(std::memory_order_relaxed);
    if (c > 0) return c;
  }
  int n = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    n = 256;
  if (dev < 64) cache[dev].store(n, std::memory_order_relaxed);
  return n;
}

// How the items are cut and dealt: R ranges of the chunk list, and xq (see
// split_slot).  The pair that makes the longest sequence of items on one block
// shortest, taking every document as its nch chunks (an item counts its chunk
// groups and half a group more), and more where an XCD would draw on the memory
// behind its L2 faster than it delivers: per K slice, the chunks of the ranges
// that it holds together and the rows of its query groups.  Of the R that give an
// XCD the same number of ranges only the groups differ, so the largest stands for
// all (and the smallest with its groups is taken): a quarter of the R or less is
// looked at (512 x 512, fp32, host time 21 us each R, 5.5 so, the same cuts).
struct SplitCut {
  int R, xq;
};
SplitCut split_cut(int nqg, int Bd, int nch, int xcd_blocks, int cg, bool f32) {
  constexpr double kXcdBytesPerUs = 0.7e6;                // memory bandwidth share of an XCD
  const double slice_us = f32 ? 6.1 : 0.77;               // a block's MFMAs per slice at 2 GHz
  const int docch = std::max(nch, 1);
  auto groups_of = [&](int R) { return ((int64_t)((Bd + R - 1) / R) * docch + cg - 1) / cg; };
  SplitCut best{1, 8};
  double best_cost = 0.0;
  for (int xq = 1; xq <= kSpXcds; xq *= 2) {
    const int xr = kSpXcds / xq, nqx = (nqg + xq - 1) / xq;
    const int rmax = std::min(Bd, xr * xcd_blocks * 2);
    for (int nrx = 1; (nrx - 1) * xr < rmax; ++nrx) {
      const int R = std::min(nrx * xr, rmax);
      const int64_t passes = ((int64_t)nqx * nrx + xcd_blocks - 1) / xcd_blocks;
      const int held_r = std::min(nrx, xcd_blocks);
      const int held_q = std::min(nqx, std::max(1, xcd_blocks / nrx));
      const double bytes = (double)(held_r * cg + held_q * kRows) * kTile * kSliceBytes;
      const double cost = (double)passes * ((double)groups_of(R) + 0.5) *
                          std::max(1.0, bytes / slice_us / kXcdBytesPerUs) * (1.0 + 1e-9 * bytes);
      if (best_cost == 0.0 || cost < best_cost) {
        best = SplitCut{R, xq};
        best_cost = cost;
      }
    }
  }
  const int xr = kSpXcds / best.xq;
  const int64_t groups = groups_of(best.R);
  while ((best.R - 1) % xr != 0 && groups_of(best.R - 1) == groups) --best.R;
  return best;
}

}  // namespace

// Tokens in one run (kFlat) where that saves a fifth of the query groups, up to 8
// of them counted as the power of two that the XCDs are dealt: less is used up
// by the token maxima's way through memory and the sum's launch (fp32, d = 64, 60 x
// 60: 8 groups 50 us, as 5 groups of one run 53, as 4 37), and where there is work to
// save (bf16, d = 256, 30 x 30: 4 groups 18.8 us, as 2 22.5).  The maxima's array is
// bounded, and a tile's tape entries lie within 2^30 bytes.
SplitRows split_rows(int64_t Bq, int64_t Tq, int64_t Bd) {
  SplitRows r;
  r.ntq = Tq > kTile ? (Tq + kTile - 1) / kTile : 1;
  r.nqg = (Bq * r.ntq + kRows - 1) / kRows;
  const int64_t ntok = Bq * Tq, ftiles = (ntok + kTile - 1) / kTile;
  const int64_t fgroups = (ftiles + kRows - 1) / kRows;
  auto dealt = [](int64_t n) { return n <= 2 ? n : n <= 4 ? 4 : n <= kSpXcds ? kSpXcds : n; };
  r.flat = dealt(fgroups) * 5 <= dealt(r.nqg) * 4 && r.nqg * Bd >= 256 && ntok <= ((int64_t)1 << 30) &&
           (Tq + kTile) * Tq < 65536 && ftiles * kTile * Bd <= ((int64_t)1 << 26) &&
           (kTile + 1) * Bd * Tq < ((int64_t)1 << 28);
  if (r.flat) {
    r.ntq = ftiles;
    r.nqg = fgroups;
  }
  // One run stores token maxima whatever its tiles (32 tokens in all are one).
  r.stored = r.flat ? ftiles * kTile * Bd : r.ntq > 1 ? Bq * r.ntq * Bd : 0;
  return r;
}

hipError_t launch_inbatch_split(int32_t dtype, const InBatchSplitArgs& args_in,
                                hipStream_t stream) {
  InBatchSplitArgs A = args_in;
  const int Bq = A.Bq, Tq = A.Tq;
  const SplitRows rows = split_rows(Bq, Tq, A.Bd);
  const bool flat = rows.flat;
  A.ntq = (int)rows.ntq;
  A.nqg = (int)rows.nqg;
  if (flat) {
    A.qtok = Tq;
    A.qrecip = (65536u + (unsigned)Tq - 1) / (unsigned)Tq;
    A.Bq = 1;
    A.Tq = Bq * Tq;
  }
  // kBlocks blocks per CU (CUs a multiple of 8, so slot x stays on XCD x % 8).
  const int cus = std::max(kSpXcds, device_cus() / kSpXcds * kSpXcds);
  const int per_cu = dtype == 0 ? SplitShape<4>::kBlocks : SplitShape<2>::kBlocks;
  const int cg = dtype == 0 ? SplitShape<4>::kCg : SplitShape<2>::kCg;
  const int nch = A.Td > 0 ? (A.Td + kTile - 1) / kTile : 0;
  const SplitCut cut = split_cut(A.nqg, A.Bd, nch, cus * per_cu / kSpXcds, cg, dtype == 0);
  A.R = cut.R;
  A.xq = cut.xq;
  const int xr = kSpXcds / A.xq;
  A.nslots = kSpXcds * ((A.nqg + A.xq - 1) / A.xq) * ((A.R + xr - 1) / xr);
  // Ranges of few documents are cut by their number: cut by chunks, one of them
  // could hold two long documents and its neighbour none.
  const int by_docs = A.Bd < 4 * A.R ? 1 : 0;
  // One workspace: the plan words (documents' chunk words, then query rows'
  // words), the chunk list, the ranges, the list blocks' counts, then the tile
  // scores or token maxima St.
  const int64_t ndw = (int64_t)A.Bd * nch, nwords = ndw + (int64_t)A.Bq * A.ntq;
  auto al = [](size_t v) { return (v + 255) / 256 * 256; };
  const size_t plan_bytes = al((size_t)nwords * sizeof(uint32_t));
  const size_t list_bytes = al((size_t)A.Bd * std::max(nch, 1) * sizeof(uint4));
  const size_t rs_bytes = al((size_t)(A.R + 1 + kSpXcds) * sizeof(int32_t));  // (slots past R look there)
  const int list_blocks = (A.Bd + kListThreads - 1) / kListThreads;
  const size_t counts_bytes = list_blocks > 1 ? al((size_t)list_blocks * sizeof(int32_t)) : 0;
  const size_t st_bytes = (size_t)rows.stored * sizeof(float);
  void* ws = nullptr;
  hipError_t e = workspace_alloc(&ws, plan_bytes + list_bytes + rs_bytes + counts_bytes + st_bytes, stream);
  if (e != hipSuccess) return e;
  uint32_t* const plan = static_cast<uint32_t*>(ws);
  uint4* const list = reinterpret_cast<uint4*>(static_cast<char*>(ws) + plan_bytes);
  int32_t* const rs = reinterpret_cast<int32_t*>(static_cast<char*>(ws) + plan_bytes + list_bytes);
  int32_t* const counts = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(rs) + rs_bytes);
  A.qwords = plan + ndw;
  A.list = list;
  A.rs = rs;
  if (st_bytes > 0)
    A.St = reinterpret_cast<float*>(reinterpret_cast<char*>(counts) + counts_bytes);
  hipLaunchKernelGGL(split_plan_kernel, dim3((unsigned)std::min<int64_t>((nwords + 7) / 8, 1024)),
                     dim3(256), 0, stream, A.dm, A.qm, A.Bd, A.Td, nch, A.Bq, A.Tq, A.ntq, plan);
  if (list_blocks > 1)
    hipLaunchKernelGGL(split_count_kernel, dim3((unsigned)list_blocks), dim3(kListThreads), 0, stream, plan,
                       A.Bd, nch, counts);
  hipLaunchKernelGGL(split_list_kernel, dim3((unsigned)list_blocks), dim3(kListThreads), 0, stream, plan,
                     A.Bd, nch, A.R, by_docs, counts, list, rs);
  e = hipGetLastError();
  const dim3 grid((unsigned)std::min(A.nslots, cus * per_cu)), block(64 * kSpWaves);
  if (e == hipSuccess) {
    auto go = [&](auto op, auto whole, auto tape, auto fl) {
      hipLaunchKernelGGL((inbatch_split<decltype(op), decltype(whole)::value, decltype(tape)::value,
                                        decltype(fl)::value>),
                         grid, block, 0, stream, A);
    };
    auto by_flat = [&](auto op, auto whole, auto tape) {
      if (flat) go(op, whole, tape, std::true_type());
      else go(op, whole, tape, std::false_type());
    };
    auto by_tape = [&](auto op, auto whole) {
      if (A.args) by_flat(op, whole, std::true_type());
      else by_flat(op, whole, std::false_type());
    };
    auto by_whole = [&](auto op) {
      if (A.rowbytes % kSliceBytes == 0) by_tape(op, std::true_type());
      else by_tape(op, std::false_type());
    };
    if (dtype == 1) by_whole(OpF16());
    else if (dtype == 2) by_whole(OpBF16());
    else by_whole(OpF32());
    e = hipGetLastError();
  }
  if (e == hipSuccess && flat) {
    hipLaunchKernelGGL(split_token_sum_kernel,
                       dim3((unsigned)std::min<int64_t>(((int64_t)Bq * A.Bd + 255) / 256, 8192)), dim3(256), 0,
                       stream, A.St, (int64_t)A.ntq * kTile, Bq, A.Bd, A.qm, Tq, A.norm, A.S);
    e = hipGetLastError();
  } else if (e == hipSuccess && A.ntq > 1) {
    hipLaunchKernelGGL(split_tile_sum_kernel,
                       dim3((unsigned)std::min((A.Bd + 255) / 256, 64),
                            (unsigned)std::min(A.Bq, 65535)),
                       dim3(256), 0, stream, A.St, A.ntq, A.Bq, A.Bd, A.qm, A.Tq, A.norm, A.S);
    e = hipGetLastError();
  }
  const hipError_t ef = workspace_free(ws, stream);
  if (e == hipSuccess) e = ef;
  return e;
}

}  // namespace fms
