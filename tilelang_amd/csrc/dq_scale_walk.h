// Where the direct-to-LDS GEMM (dq_gemm_core.h) finds a row's scales: 16-bit groups that travel a dword per row at a time, two
// groups each, into a ring of four slots.  Plain arithmetic, so that the host can check it.
//
// Rows of an odd count of groups: every other row starts in the middle of a dword.  Dword i of such a row holds groups
// 2 i - 1 and 2 i; it is asked for one ahead, where dword i - 1 of the rows between them is, so that both kinds of row have
// a group by the time that its tile is due, and dword 0 goes before all others to the slot that is needed last.
#pragma once

#ifdef __HIPCC__
#define DQ_HD __host__ __device__ __forceinline__
#else
#define DQ_HD inline
#endif

namespace dq {
namespace gemm {

struct ScaleWalk {
  unsigned start, ahead;  // byte offsets: dword 0 of the row, and what is asked for with dword 0 of the rows that are not ahead
  int last;               // odd counts: the index of the last group's dword in the rows that are not ahead; else -1

  DQ_HD ScaleWalk(unsigned row, unsigned groups, bool odd) {
    const unsigned at = row * groups * 2;
    start = at & ~3u;
    ahead = start + 4u * (at >> 1 & 1);
    last = odd ? (int)(groups >> 1) : -1;
  }
  // From which byte, less 4 * dword, the four bytes of index `dword` come.  With the last dword the rows ahead have had all of
  // theirs; of the others its second half is the next row's, so an odd count of groups goes with an even count of rows.
  DQ_HD unsigned from(int dword) const { return dword == last ? start : ahead; }
  // The byte in the ring (slots of 1024) at which a group lies, of a row that is not ahead and of one that is
  static DQ_HD int aligned(int group) { return ((group >> 1) & 3) * 1024 + (group & 1) * 2; }
  static DQ_HD int one_ahead(int group) { return (((group - 1) >> 1) & 3) * 1024 + ((group + 1) & 1) * 2; }
};

}  // namespace gemm
}  // namespace dq
