// fms_few.hpp -- the scan with one workgroup per pair: few pairs, and fp32.
//
// The other scans give a pair to one wave, which walks the document's chunks
// one after the other: with fewer pairs than the chip has wave slots most of
// it idles while each wave pays every chunk's memory latency and MFMA chain
// in series (64 fp32 pairs of 32 x 180 tokens, d = 128: 89 us, of which 10 us
// are the wave's 384 MFMAs).  Here the waves of a workgroup share one pair: wave w takes
// chunks w, w + W, ..., keeps its own running max / argmax over them, and the
// first wave merges the W results through LDS once per query tile.
#pragma once

#include "fms_scan.hpp"

namespace fms {

constexpr int kFewMaxWaves = 8;

// One 32-byte column group m of 32 rows: lane (r32, h) holds the 16 bytes of
// row r32 at 32 m + 16 h.  For 16-bit and INT8 features that is one MFMA
// operand.  For fp32 it is four (features 8m + 4h .. + 3): a lane's dwords
// pair up across the wave halves by two permlane32 swaps, after which the
// four registers are the k-blocks (8m, 8m+1), (8m+4, 8m+5), (8m+2, 8m+3),
// (8m+6, 8m+7) with the lower feature in the lower half, the operands the
// dword loads of the other fp32 scans give.
__device__ __forceinline__ void few_pair_halves(u32x4& x) {
  const auto p = __builtin_amdgcn_permlane32_swap(x[0], x[1], false, false);
  const auto q = __builtin_amdgcn_permlane32_swap(x[2], x[3], false, false);
  x = u32x4{p[0], p[1], q[0], q[1]};
}

// acc0 (even k-blocks) and, with kTwo, acc1 (odd ones) += the products of
// column group m, in the k order of the other scans.
template <class Op, bool kTwo>
__device__ __forceinline__ void few_mma(u32x4 a, u32x4 b, int m, typename Op::Acc& acc0,
                                        typename Op::Acc& acc1) {
  if constexpr (Op::kEsz == 4) {
    few_pair_halves(a);
    few_pair_halves(b);
    typename Op::Acc& odd = kTwo ? acc1 : acc0;
    acc0 = Op::mma(a[0], b[0], acc0);
    odd = Op::mma(a[2], b[2], odd);
    acc0 = Op::mma(a[1], b[1], acc0);
    odd = Op::mma(a[3], b[3], odd);
  } else if constexpr (kTwo) {
    if (m & 1) acc1 = Op::mma(a, b, acc1);
    else acc0 = Op::mma(a, b, acc0);
  } else {
    acc0 = Op::mma(a, b, acc0);
  }
}

// kB column groups of row r (byte offset `row` of the row), from group m0 on;
// groups past the row read out of range (zeros).
template <int kB>
__device__ __forceinline__ void few_load(u32x4 (&f)[kB], rsrc_t r, int row, int m0, int h,
                                         int rowbytes) {
#pragma unroll
  for (int i = 0; i < kB; ++i) {
    const int o = (m0 + i) * 32 + h * 16;
    const int past = -(int)(o >= rowbytes) & 0x7fffffff;
    f[i] = buf_load16(r, (row + o) | past);
  }
}

// What a wave found over its chunks, per query token: the best score and its
// token (0: none above -inf), and its first valid row's score and token.
struct FewPart {
  float mx;
  int tok;
  float first;
  int ftok;
};

// The scan position of this workgroup.  In document order an XCD takes a run of
// consecutive positions (workgroups are dealt to the XCDs round-robin), so the
// pairs that share a document meet in one L2 while it is there.
template <class L>
__device__ __forceinline__ int64_t few_position(int64_t npairs) {
  const int64_t b = blockIdx.x;
  if constexpr (interleaved<L>::value) {
    const int64_t x = b & 7, k = b >> 3, each = npairs >> 3, more = npairs & 7;
    return x * each + (x < more ? x : more) + k;
  }
  return b;
}

// kB: column groups in flight per operand.  kOne: a row is at most kB groups,
// so the query tile is loaded once per tile instead of per chunk.  kTwo: even
// and odd k-blocks accumulate apart and are added at the chunk's end, as
// scan_split does for the dims it serves; results are those of the scan that
// would take the call with more pairs, bit for bit.
template <class Op, class L, int kB, bool kOne, bool kTwo>
__global__ void __launch_bounds__(64 * kFewMaxWaves) __attribute__((amdgpu_waves_per_eu(4)))
scan_few(const ScanArgs<L> A) {
  typedef typename Op::Acc Acc;
  __shared__ FewPart part[2][kFewMaxWaves][kTile];
  const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
  const int w = uniform((int)(threadIdx.x >> 6)), W = uniform((int)(blockDim.x >> 6));
  const PairView v = uniform_view(A.lay.get(few_position<L>(A.npairs)));
  const int rowbytes = A.dim * Op::kEsz;
  const int nm = (rowbytes + 31) / 32;
  const int nch = (v.td + kTile - 1) / kTile;
  const rsrc_t rq = make_rsrc_u(v.q, (uint32_t)v.tq * (uint32_t)rowbytes);
  const rsrc_t rd = make_rsrc_u(v.d, (uint32_t)v.td * (uint32_t)rowbytes);
  float score = 0.0f;
  for (int qt = 0; qt < A.nqt; ++qt) {
    const int t = qt * kTile + r32;
    u32x4 b[kB];
    if constexpr (kOne) few_load<kB>(b, rq, t * rowbytes, 0, h, rowbytes);
    float qscale = 0.0f;
    if constexpr (Op::kInt) qscale = load_qscale(v, t);
    float mx = -INFINITY, first = -INFINITY;
    int slot = -1, fslot = -1;
    for (int ch = w; ch < nch; ch += W) {
      const int row = ch * kTile + r32;
      uint32_t mbyte = 1u;
      if (v.dm) mbyte = buf_load1(make_rsrc_u(v.dm, (uint32_t)v.td), row);
      const uint32_t m32 = chunk_rows_valid(v, ch, r32, mbyte);
      if (m32 == 0u) continue;  // no valid row: nothing to read
      float ds[1];
      load_ds<Op>(ds, v, ch, r32);
      Acc acc0 = {}, acc1 = {};
      for (int m0 = 0; m0 < (kOne ? 1 : nm); m0 += kB) {
        u32x4 a[kB];
        few_load<kB>(a, rd, row * rowbytes, m0, h, rowbytes);
        if constexpr (!kOne) few_load<kB>(b, rq, t * rowbytes, m0, h, rowbytes);
#pragma unroll
        for (int i = 0; i < kB; ++i) few_mma<Op, kTwo>(a[i], b[i], i, acc0, acc1);
      }
      if constexpr (kTwo) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc0[r] += acc1[r];
      }
      float s[16];
      acc_to_scores<Op>(acc0, qscale, ds, h, s);
      take_first_row(s, m32, h, ch, first, fslot);
      update_chunk(s, m32, h, ch, mx, slot);
    }
    int tok = slot_to_token(slot, h);
    merge_halves(mx, tok, h);
    int ftok = slot_to_token(fslot, h);
    const int otok = (int)lane_xor32((uint32_t)ftok, h);
    const float ofirst = __builtin_bit_cast(float, lane_xor32(__builtin_bit_cast(uint32_t, first), h));
    first = ftok != 0 ? first : ofirst;  // one half holds the wave's first valid row
    ftok = ftok != 0 ? ftok : otok;
    FewPart(&P)[kFewMaxWaves][kTile] = part[qt & 1];
    if (h == 0) P[w][r32] = FewPart{mx, tok, first, ftok};
    __syncthreads();  // (one per tile: the next tile writes the other half of `part`)
    if (w == 0) {
      for (int i = 1; i < W; ++i) {
        const FewPart o = P[i][r32];
        const bool take = o.tok != 0 && (tok == 0 || o.mx > mx || (o.mx == mx && o.tok < tok));
        mx = take ? o.mx : mx;
        tok = take ? o.tok : tok;
        const bool ftake = o.ftok != 0 && (ftok == 0 || o.ftok < ftok);
        first = ftake ? o.first : first;
        ftok = ftake ? o.ftok : ftok;
      }
      // The document's first valid row stands when it is NaN or when nothing
      // exceeds -inf (see take_first_row); otherwise it was folded with the rest.
      const bool keep_first = ftok != 0 && (tok == 0 || is_nan_bits(first));
      mx = keep_first ? first : mx;
      tok = keep_first ? ftok : tok;
      uint32_t qmb = 1u;
      if (v.qm) qmb = buf_load1(make_rsrc_u(v.qm, (uint32_t)v.tq), t);
      const bool tvalid = t < v.tq && qmb != 0u;
      const float p = (tvalid && tok != 0) ? mx : 0.0f;
      if (h == 0 && t < A.rows) {
        const int64_t o = v.out * (int64_t)A.rows + t;
        if (A.args) A.args[o] = tvalid ? tok : 0;
        if (A.partial) A.partial[o] = p;
      }
      score += half_sum(p);
    }
  }
  if (w == 0) write_score(A, v, score, lane);
}

// Chunks a pair's document has on average (the host knows padded lengths and
// the size of a ragged store, not each ragged document's length).
inline int64_t few_chunks(const LayPaired& l, int64_t) { return ((int64_t)l.Td + kTile - 1) / kTile; }
inline int64_t few_chunks(const LayCand& l, int64_t) { return ((int64_t)l.Td + kTile - 1) / kTile; }
inline int64_t few_chunks(const LayCandSorted& l, int64_t n) { return few_chunks(l.c, n); }
inline int64_t few_chunks(const LayPacked& l, int64_t n) { return l.ntok / (n * kTile) + 1; }
inline int64_t few_chunks(const LayVarlen& l, int64_t n) { return l.nd / (n * kTile) + 1; }

// Most pairs of a call that take a workgroup each.  16-bit and INT8: a wave's
// fragment loads touch 32 rows each, and with every wave loading its own query
// tile that sets the pace once the chip is full, so two workgroups per CU are
// the most that pay (d = 128, Td = 180, us per call at 512 / 1000 / 2000 pairs:
// 9.3 / 15.8 / 29.5 here, 10.5 / 12.5 / 18.6 with a wave per pair; 64 documents
// of 900 tokens 11.6 against 28.1, 1000 of them 44 against 35).  fp32: at any
// count, since the other scans load dwords (16 bytes per lane here): 64 pairs
// 9.9 against 88.7 us, 2000 58 against 176; the bound there is the grid's
// 32-bit work-item count.  Documents of one chunk leave nothing to share and stay
// with the other scans, in fp32 too, where the loads alone would be worth a
// workgroup from d = 64 on (2000 pairs of 32 x 32 tokens, d = 128: 15 against 44 us;
// d = 32 within a tenth).
template <class Op>
constexpr int64_t few_pairs() {
  return Op::kEsz == 4 ? (int64_t)1 << 22 : 512;
}

// Past one workgroup per CU, 16-bit rows that are not kept (every chunk loads the query
// tile again) compete with scan_fast at d = 256 and scan_split, which keep or stream it:
// bytes of a document, on average, up to which a workgroup per pair still pays.
// us per call at 512 pairs, wave / workgroup per pair: packed documents (one query,
// whose lines all workgroups read at once), d = 256, up to 180 / 400 / 2000 tokens 16 / 14,
// 27 / 27, 105 / 158; d = 768, 90 / 900 / 2000 tokens 21 / 24, 153 / 255, 334 / 582; pairs
// with a query each, d = 256, 900 / 2000 tokens 68 / 62, 163 / 180 (ragged, 666 .. 2000
// tokens 106 / 153), d = 768 417 / 290, 902 / 638.  (At 256 pairs the workgroups win
// throughout, 1.1 to 4 times.)
constexpr int64_t kFewFull = 256;
template <class L>
constexpr int64_t few_doc_bytes(bool) { return 0; }
template <>
constexpr int64_t few_doc_bytes<LayPacked>(bool split) { return split ? 48 << 10 : 96 << 10; }
template <>
constexpr int64_t few_doc_bytes<LayPaired>(bool split) { return split ? INT64_MAX : 512 << 10; }
template <>
constexpr int64_t few_doc_bytes<LayCand>(bool split) { return few_doc_bytes<LayPaired>(split); }
template <>
constexpr int64_t few_doc_bytes<LayVarlen>(bool split) { return few_doc_bytes<LayPaired>(split); }

// 16-byte fragment loads: every row is whole 16-byte units from an aligned base
// (fp32 scans otherwise load dwords and ask for neither).
inline bool few_aligned(const void* q, const void* d) {
  return ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(d)) & 15u) == 0;
}
inline bool few_aligned(const LayPaired& l) { return few_aligned(l.Q, l.D); }
inline bool few_aligned(const LayCand& l) { return few_aligned(l.Q, l.G); }
inline bool few_aligned(const LayCandSorted& l) { return few_aligned(l.c); }
inline bool few_aligned(const LayPacked& l) { return few_aligned(l.q, l.tok); }
inline bool few_aligned(const LayVarlen& l) { return few_aligned(l.Qt, l.Dt); }

// The launch, or false when the call stays with the wave-per-pair scans.
// two: the scan that serves this dim with more pairs is scan_split, which keeps two
// chains; fast: it is scan_fast.
template <class Op, class L>
bool launch_few(const ScanArgs<L>& A, bool vec, bool two, bool fast, hipStream_t stream, hipError_t* err) {
  const int rowbytes = A.dim * Op::kEsz;
  if (!vec || A.dim <= 0 || rowbytes % 16 != 0 || A.npairs < 1 || A.npairs > few_pairs<Op>()) return false;
  if (!few_aligned(A.lay)) return false;
  const int64_t nch = few_chunks(A.lay, A.npairs);
  if (nch < 2) return false;
  const unsigned W = (unsigned)(nch < kFewMaxWaves ? nch : kFewMaxWaves);
  const dim3 grid((unsigned)A.npairs), block(64 * W);
  const int nm = (rowbytes + 31) / 32;
  if (Op::kEsz == 2 && A.npairs > kFewFull && nm > 8 && (two || fast) &&
      nch * kTile * rowbytes > few_doc_bytes<L>(two))
    return false;
  if constexpr (Op::kEsz == 4) {
    if (two && nm <= 8)
      hipLaunchKernelGGL((scan_few<Op, L, 8, true, true>), grid, block, 0, stream, A);
    else if (two)
      hipLaunchKernelGGL((scan_few<Op, L, 8, false, true>), grid, block, 0, stream, A);
    else
      hipLaunchKernelGGL((scan_few<Op, L, 8, false, false>), grid, block, 0, stream, A);
  } else {
    if (two)
      hipLaunchKernelGGL((scan_few<Op, L, 8, false, true>), grid, block, 0, stream, A);
    else if (nm <= 4)
      hipLaunchKernelGGL((scan_few<Op, L, 4, true, false>), grid, block, 0, stream, A);
    else if (nm <= 8)
      hipLaunchKernelGGL((scan_few<Op, L, 8, true, false>), grid, block, 0, stream, A);
    else
      hipLaunchKernelGGL((scan_few<Op, L, 8, false, false>), grid, block, 0, stream, A);
  }
  *err = hipGetLastError();
  return true;
}

}  // namespace fms
