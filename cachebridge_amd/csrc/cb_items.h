// Items of the support kernel: which XCD maps which job over which tokens.
// Integer bookkeeping without device code, so that a host program can walk the
// same lists (tests/test_items.py).
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define CB_ITEMS_FN __host__ __device__ __attribute__((always_inline)) inline
#else
#define CB_ITEMS_FN inline
#endif

constexpr int kSupTile = 256;      // tokens per item
constexpr int kSupJobGroup = 16;   // jobs of an XCD that run interleaved, chunk by chunk

// Host: class c of a launch whose items hold at most `chunk` tokens; returns
// its chunks per job. A class without tokens has none: its jobs have no items.
template <class Args>
inline int64_t set_class_tokens(Args& a, int c, int64_t first, int64_t count, int chunk) {
  const int64_t nch = (count + chunk - 1) / chunk;
  a.cls_tok_first[c] = static_cast<int32_t>(first);
  a.cls_tok_count[c] = static_cast<int32_t>(count);
  a.cls_nchunks[c] = static_cast<int32_t>(nch);
  return nch;
}

// XCD x takes units x, x + 8, ... of each class (the plan orders the units so
// that these are a run of adjacent keys jobs and a run of adjacent values jobs
// in the sorted job order, whose support lists share source layers) and runs
// them in groups of kSupJobGroup jobs, the group's jobs interleaved per token
// chunk, so that the items an XCD runs at one time read overlapping source
// rows and share its L2. Item p of its list (job_of: the job of a unit), false
// past the end.
struct SupItem {
  int job, lo, hi;  // tokens [lo, hi)
};

template <class Args, class JobOf>
CB_ITEMS_FN bool support_list_item(const Args& a, int x, int64_t p, JobOf&& job_of, SupItem& it) {
  for (int c = 0; c < a.ncls; ++c) {
    const int nj = a.cls_unit_end[c] - a.cls_unit_begin[c];
    const int mine = nj > x ? (nj - x + 7) / 8 : 0;
    const int nch = a.cls_nchunks[c];
    const int64_t count = static_cast<int64_t>(mine) * nch;
    if (p < count) {
      const int64_t gsz = static_cast<int64_t>(kSupJobGroup) * nch;
      const int g = static_cast<int>(p / gsz);
      const int r = static_cast<int>(p - g * gsz);
      const int left = mine - g * kSupJobGroup;
      const int gj = kSupJobGroup < left ? kSupJobGroup : left;
      const int ch = r / gj, jl = g * kSupJobGroup + (r - ch * gj);
      it.job = job_of(a.cls_unit_begin[c] + x + 8 * jl);
      it.lo = a.cls_tok_first[c] + ch * kSupTile;
      const int end = a.cls_tok_first[c] + a.cls_tok_count[c];
      it.hi = it.lo + kSupTile < end ? it.lo + kSupTile : end;
      return true;
    }
    p -= count;
  }
  return false;
}
