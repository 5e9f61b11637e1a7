// rate_search.h -- which codes a bitplane's rate search tries and what the run
// records say about them; no GPU needed, so host tests compile it by itself.
#pragma once
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define DVC_RATE_FN __host__ __device__ inline
#else
#define DVC_RATE_FN inline
#endif

namespace dvc {

// DYNAMICSTEP rate search (LdpcaDecoder.cpp:19-21, 669-672, 760-768): after
// the r-th failed request (r = 0, 1, ...) the search moves 1 + {0,1,2,3}[min(r,3)]
// codes up, so it tries the codes start + 0, 1, 3, 6, 10, 14, 18, ... below
// the full rate, then the full rate.
DVC_RATE_FN bool dynstep_tries(int off) {
  return off == 0 || off == 1 || off == 3 || off == 6 || (off >= 10 && (off - 10) % 4 == 0);
}
// The offset from the start code tried after offset `off` fails.
DVC_RATE_FN int dynstep_next(int off) {
  return off < 1 ? 1 : off < 3 ? 3 : off < 6 ? 6 : off < 10 ? 10 : off + 4;
}

// Status of a run record (its second word).
enum { REC_FAILED = 0, REC_CRC_MISMATCH = 1, REC_ACCEPTED = 2, REC_CANCELLED = 3, REC_NOT_RUN = -1 };

// The accepted code is the search's only if every code it tries before that one
// has run to its end and failed; a launch that ended early (a split launch that
// gave up waiting) leaves some without such a record.  Returns the first of
// those codes, or -1.  rec: one record per code (.y is the status).
template <class Record>
inline int unfinished_code(const Record *rec, int start, int accepted, int rate_step) {
  for (int l = start; l < accepted; l++) {
    if (rate_step && !dynstep_tries(l - start)) continue;
    if (rec[l].y != REC_FAILED && rec[l].y != REC_CRC_MISMATCH) return l;
  }
  return -1;
}

}  // namespace dvc
