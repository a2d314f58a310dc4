// fms_inbatch_split.hpp -- launcher of the split-K InBatch() kernel (the
// feature dim taken a K slice at a time): 16-bit features with dims the
// register-resident kernel does not take, and fp32 features.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fms {

struct InBatchSplitArgs {
  const char* Q;      // (Bq, Tq, dim) features
  const char* D;      // (Bd, Td, dim)
  const uint8_t* qm;  // (Bq, Tq) nullable
  const uint8_t* dm;  // (Bd, Td) nullable
  float* S;           // (Bq, Bd): S[i*Bd + j] = MaxSim(Q_i, D_j)
  int32_t* args;      // (Bq, Bd, Tq) nullable
  int Bq, Bd, Tq, Td;
  int rowbytes;       // dim * element bytes (a multiple of 16)
  int norm = 0;
  // filled by the launcher: query rows are 32-token tiles, ntq per query
  // (scored into St (Bq * ntq, Bd) and summed into S when ntq > 1); nqg
  // groups of 8 query rows
  int ntq = 1, nqg = 1;
  float* St = nullptr;
  // filled by the launcher when tiles are cut from all queries' tokens as one run:
  // tokens of a query (Bq is then 1, Tq all tokens, St token maxima (Bd, 32 * ntq))
  int qtok = 0;
  uint32_t qrecip = 0;  // ceil(2^16 / qtok)
  // filled by the launcher: valid tokens of every query row, the list of
  // document chunks (see split_list_kernel), the first entry of each of its R
  // ranges, and the number of block-order slots (see split_slot)
  const uint32_t* qwords = nullptr;
  const uint4* list = nullptr;
  const int32_t* rs = nullptr;
  int R = 1, xq = 8;
  int nslots = 0;
};

// Element bytes 2 or 4; rows a multiple of 16 bytes; 16-byte aligned bases.
bool inbatch_split_supported(int esz, int64_t dim, int64_t Tq, int64_t Td, int64_t Bq,
                             int64_t Bd, const void* Q, const void* D);
// The query rows of a call: one run of all tokens (flat) or tiles per query, ntq
// tiles (flat: in all) in nqg groups of 8, and the floats of St (0: scores go
// straight to S).
struct SplitRows {
  bool flat = false;
  int64_t ntq = 1, nqg = 1, stored = 0;
};
SplitRows split_rows(int64_t Bq, int64_t Tq, int64_t Bd);
// dtype: 0 fp32, 1 fp16, 2 bf16 (the C ABI's codes).
hipError_t launch_inbatch_split(int32_t dtype, const InBatchSplitArgs& args, hipStream_t stream);

}  // namespace fms
