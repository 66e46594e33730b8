// Work-groups of one pass of the chunked ILU's apply, in plain C++.
#pragma once
#ifdef __HIPCC__
#define SG_HD __host__ __device__
#else
#define SG_HD
#endif

namespace sg {

struct PassGroup {
  int chunk, group;  // column group `group` of chunk `chunk` (which may not exist)
};

// What work-group `block` of a pass solves, with ng column groups a chunk.
// Work-groups are dealt to the 8 XCDs round-robin by index and started there in
// that order.  The groups of a chunk sit on one XCD, in the order in which the
// pass hands their edge values on: a group's source is started before it, so in
// a launch of one pass a waiting group's source has run or is running, however
// few work-groups the chip has room for.
SG_HD inline PassGroup pass_group(int block, int ng, bool ascending) {
  const int xcd = block & 7, slot = block >> 3, nth = slot % ng;
  return {slot / ng * 8 + xcd, ascending ? nth : ng - 1 - nth};
}
SG_HD inline int pass_blocks(int nchunk, int ng) { return (nchunk + 7) / 8 * 8 * ng; }

}  // namespace sg
