// Host side of the sync-free sweeps: what is decided from a factor's structure
// alone (no device code).
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace bcm {

// Strips (k_sweep_strip): block sizes up to 16 rows, four lanes each. (At 24,
// with the layout of k_sweep_free, a row's factor values did not fit the
// registers twice: 17 x 16 x 15 took 186 us by levels, 162 to 218 us in strips,
// a periodic 16^3 cell 108 against 179.)
constexpr int kStripBlock = 16;
// Waves of a strip, and dependency blocks of a row held in registers (twice,
// for the next row): in that layout 20 x 20 x 20 x block 8 took 136 us with 8
// waves, 127 with 16; 20 x 19 x 18 x block 12 (FP64) 166 and 220, block 16 120
// and 203.
constexpr int strip_waves(int b) { return b <= 9 ? 16 : 8; }
constexpr int strip_held(int b) { return b >= 16 ? 3 : 4; }

// How many strips ns rows are cut into: 16 rows a strip, up to one strip per
// compute unit; a strip's values within 48 KB of LDS. (64 x 64 heat, block 9,
// both sweeps: 448 us by levels; strips of 16, 32, 64 rows: 244, 249, 254 us.)
inline int strip_count(int b, int ns) {
  const int64_t bytes = (int64_t)ns * b * 8, lds = 48 << 10;
  return (int)std::max<int64_t>(std::min(256, ns / 16), (bytes + lds - b * 8 - 1) / (lds - b * 8));
}

// Whether nrhs columns of a sweep over ns rows in `levels` levels, factor values
// of `bytes` bytes, run in strips rather than level by level on all waves
// (k_sweep_free). Both sides in us, both sweeps of a preconditioner, strips
// first:
// * A strip does one or two rows at a time, so it must not have many of a
//   level: 256 strips of 3D grids win up to 40 rows a level for every row of
//   the block. Block 6: 239 rows 478 / 515, 317 rows 675 / 583. Block 9: 255
//   rows 498 / 488, 386 rows 290 / 321. Block 12: 300 rows 243 / 363, 481 rows
//   437 / 475. Block 3: 158 rows 4142 / 4185, 221 rows 7619 / 5734.
// * Long strips pass from line to line of a 2D grid late. Block 9, 625 rows a
//   strip: 2478 / 2729; block 3, 1914 rows: the case above. Their factor values
//   come from beyond the caches: 200 x 200 x block 12 (156 rows, 180 KB of
//   diagonal blocks a strip) 1308 / 1750, block 16 (312 KB) 1730 / 1367. Where
//   levels are as narrow as 32 rows, strips of any length win (a chain: 0.43 us a
//   level against 1.2).
// * Columns are strips of their own, with factor values of their own, while
//   columns of a row on neighbouring waves share theirs. Blocks up to 9: 478 rows
//   and columns a level 497 / 532, 717 569 / 540. Block 16, FP64: 342 267 / 307,
//   414 241 / 208; FP32: 498 1550 / 1374.
inline bool sweep_in_strips(int b, int bytes, int64_t ns, int64_t levels, int64_t nrhs) {
  if (b > kStripBlock || ns < 32 || ns > 44LL * b * levels || ns * nrhs > 512 * levels) return false;
  const int64_t block = (int64_t)b * b * bytes, strip_rows = ns / strip_count(b, (int)ns);
  if (b > 9 && ns * nrhs * block > levels * (768 << 10)) return false;
  return ns <= 32 * levels || (b <= 9 ? strip_rows <= 640 : strip_rows * block <= 256 << 10);
}

struct Strips {
  int count = 0, rows_max = 0;       // 0: none
  std::vector<int> rows, ptr, code;  // rows strip by strip, first position of each, dependencies (k_sweep_strip)
};

// Cuts the rows of a factor (dependency lists ia, ja; levels lev, `levels` of
// them) into strips: consecutive pieces of a depth-first topological order, the
// rows of each by level. No strips where more than an eighth of the rows has
// dependencies beyond those that the kernel holds, or where a single column
// takes none.
inline Strips cut_strips(int b, int bytes, int levels, const std::vector<int>& ia, const std::vector<int>& ja,
                         const std::vector<int>& lev, bool forward) {
  Strips t;
  const int ns = (int)ia.size() - 1;
  int64_t more = 0;
  for (int r = 0; r < ns; ++r) more += ia[r + 1] - ia[r] > strip_held(b) ? 1 : 0;
  if (more * 8 > ns || !sweep_in_strips(b, bytes, ns, levels, 1)) return t;
  const int P = strip_count(b, ns);
  std::vector<int> sptr(ns + 1, 0), succ(ia[ns]), cnt(ns), stack;
  for (int r = 0; r < ns; ++r) cnt[r] = ia[r + 1] - ia[r];
  for (int j = 0; j < ia[ns]; ++j) sptr[ja[j] + 1]++;
  for (int r = 0; r < ns; ++r) sptr[r + 1] += sptr[r];
  {
    std::vector<int> at(sptr.begin(), sptr.end() - 1);
    for (int q = 0; q < ns; ++q) {
      const int r = forward ? q : ns - 1 - q;
      for (int j = ia[r]; j < ia[r + 1]; ++j) succ[at[ja[j]]++] = r;
    }
  }
  for (int q = ns - 1; q >= 0; --q) {
    const int r = forward ? q : ns - 1 - q;
    if (cnt[r] == 0) stack.push_back(r);
  }
  std::vector<int>& seq = t.rows;
  seq.reserve(ns);
  while (!stack.empty()) {
    const int r = stack.back();
    stack.pop_back();
    seq.push_back(r);
    const size_t s0 = stack.size();
    for (int k = sptr[r]; k < sptr[r + 1]; ++k)
      if (--cnt[succ[k]] == 0) stack.push_back(succ[k]);
    std::reverse(stack.begin() + s0, stack.end());
  }
  std::vector<int> strip(ns), pos(ns);
  t.ptr.resize(P + 1);
  for (int k = 0; k <= P; ++k) t.ptr[k] = (int)((int64_t)ns * k / P);
  for (int k = 0; k < P; ++k) {
    std::stable_sort(seq.begin() + t.ptr[k], seq.begin() + t.ptr[k + 1],
                     [&](int x, int y) { return lev[x] < lev[y]; });
    for (int i = t.ptr[k]; i < t.ptr[k + 1]; ++i) {
      strip[seq[i]] = k;
      pos[seq[i]] = i - t.ptr[k];
    }
    t.rows_max = std::max(t.rows_max, t.ptr[k + 1] - t.ptr[k]);
  }
  t.code.resize(std::max(ia[ns], 1));
  for (int r = 0; r < ns; ++r)
    for (int j = ia[r]; j < ia[r + 1]; ++j) t.code[j] = strip[ja[j]] == strip[r] ? -1 - pos[ja[j]] : ja[j];
  t.count = P;
  return t;
}

// Bound of one dependency wait of a sweep launch, in seconds. A wave may wait
// for all of the launch that comes before its row, so the bound is a time that
// no launch takes: per level 20 us and 2 us for every dependency of a row (a
// level costs 0.65 to 4 us with rows of up to 8 dependencies, one staged chunk
// of 3 more some 1 us), 0.1 us for every block and column (0.3 to 2 ns as
// measured over whole sweeps), and 4 s for what else may hold the GPU.
// levels, deps_max and blocks of both sweeps together.
inline double sweep_wait_seconds(int64_t levels, int64_t deps_max, int64_t blocks, int64_t nrhs) {
  return 4.0 + (double)levels * (20e-6 + 2e-6 * (double)deps_max) + 1e-7 * (double)blocks * (double)nrhs;
}

}  // namespace bcm
