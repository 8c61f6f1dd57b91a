// Launch choices of the fused path on sides with a register plan, and the
// autotuner's search over them.  Host code without the GPU.
#pragma once
#include <algorithm>

namespace sf21 {

// Only choices that change launch shapes and stage order: the top-hat weight
// mode changes values and stays an explicit configuration setting.
struct TuneChoice {
  int tile = 16, K = 16, ct = 16, cw = 0, rw = 0, fp = 0;
};

inline bool wide_ok(int n) { return n == 128 || n == 256 || n == 512; }

// Column-pass variant that exists for this size and tile: 16 values per
// thread only for wide_ok sizes (tile 16 or 32), prefetching blocks only
// with tile 16 (8 values) or tile 32 (16 values).
inline int cols_variant(int n, int tile, int cw) {
  const bool wide = (cw & 1) && wide_ok(n) && (tile == 16 || tile == 32);
  const bool pipe = (cw & 2) && (tile == 16 || (wide && tile == 32));
  return (wide ? 1 : 0) | (pipe ? 2 : 0);
}

// Coordinate search from `best`, the choices in force: each dimension in turn,
// the others held at the best so far, so that the result is never slower than
// the choices it started from.  n: side, nr: radii, plane: no column and row
// passes.  timed(choice, &ms): 0, 1 (does not fit: skipped) or negative (error:
// returned at once).  Returns 1 if nothing fitted.
template <class Timed>
int tune_search(int n, int nr, bool plane, Timed&& timed, TuneChoice* best, double* best_ms) {
  bool any = false;
  int err = 0;
  auto consider = [&](const TuneChoice& t) {
    if (err) return;
    double ms;
    const int r = timed(t, &ms);
    if (r < 0) err = r;
    else if (r == 0 && (!any || ms < *best_ms)) {
      any = true;
      *best_ms = ms;
      *best = t;
    }
  };
  consider(*best);
  // larger batches read the spectrum fewer times per slice
  for (int K : {8, 12, 16, 24, 32, nr}) {
    TuneChoice t = *best;
    t.K = std::min(K, nr);
    if (t.K != best->K) consider(t);
  }
  for (int tile : {8, 16}) {
    TuneChoice t = *best;
    t.tile = tile;
    if (t.tile != best->tile) consider(t);
  }
  {
    TuneChoice t = *best;
    t.fp = 1 - t.fp;
    consider(t);
  }
  if (!plane) {
    const TuneChoice base = *best;
    const int cols[7][2] = {{8, 0}, {16, 0}, {16, 2}, {16, 1}, {16, 3}, {32, 1}, {32, 3}};
    for (auto& o : cols) {
      TuneChoice t = base;
      t.ct = o[0];
      t.cw = o[1];
      if (((o[1] & 1) && !wide_ok(n)) || (t.ct == base.ct && t.cw == base.cw)) continue;
      consider(t);
    }
    if (wide_ok(n)) {
      TuneChoice t = *best;
      t.rw = 1 - t.rw;
      consider(t);
    }
  }
  return err ? err : any ? 0 : 1;
}

}  // namespace sf21
