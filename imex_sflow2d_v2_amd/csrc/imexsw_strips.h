// imexsw_strips.h -- host arithmetic of the stencil pass's strips.
#pragma once

namespace imexsw {

// Rows per strip of whole tile columns (k_stencil): tiles_x columns of ny rows
// on `slots` resident wavefronts, a strip costing its rows and `over` more.
// The height whose rounds take least, the smallest such.  Of the heights that
// cut a column into the same number of strips only the smallest can be it, so
// about 2 sqrt(ny) heights are looked at: every launch outside a captured graph
// pays for the search (host time a launch at 2048 rows 6.3 us with every height,
// 0.9 with these; at 20000 rows 62 and 2.8).
inline int column_rows(int tiles_x, int ny, long slots, int over) {
  int best = 1;
  long cost = -1;
  for (int h = 1;;) {
    const int n = (ny + h - 1) / h;  // strips of a column
    const long t = ((long)tiles_x * n + slots - 1) / slots * (h + over);
    if (cost < 0 || t < cost) {
      cost = t;
      best = h;
    }
    if (n == 1) return best;
    h = (ny + n - 2) / (n - 1);  // the smallest height of at most n - 1 strips
  }
}

}  // namespace imexsw
