// crm_index.hpp -- grid-stride walks in 64 bits: item counts of one call may pass 2^31 (rows of a
// training batch, radiation columns times levels), and a 32-bit index that is advanced past its
// bound would wrap before that.  The same source builds for the host, so that a test can walk the
// largest counts.
#pragma once

#if defined(__HIP__)
#define CRM_INDEX_HD __host__ __device__
#else
#define CRM_INDEX_HD
#endif

// items first, first + step, ... below count
struct Strided {
  long at, step, count;
  CRM_INDEX_HD bool more() const { return at < count; }
  CRM_INDEX_HD void next() { at += step; }
};

// the tiles of `rows` rows that block `block` of `blocks` takes
CRM_INDEX_HD inline Strided tiles_of(long rows, int tile_rows, unsigned block, unsigned blocks) {
  return {(long)block, (long)blocks, (rows + tile_rows - 1) / tile_rows};
}

// the level of row `row` of (nrad, levels) rows; a 64-bit division only where it takes one
CRM_INDEX_HD inline int level_of(long row, int nrad) {
  return row >> 32 ? (int)(row / nrad) : (int)((unsigned)row / (unsigned)nrad);
}
