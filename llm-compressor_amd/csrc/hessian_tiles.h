// The order of the Hessian kernel's tiles (hessian.hip); nothing but arithmetic, so that a test can compile it for the host.
#pragma once

// Compact tile number c -> (I, J), J >= I.  Tiles are grouped into SH x SW super-tiles (as many tiles as run concurrently on
// one XCD), tiles row-major inside: workgroups sharing an L2 then touch only SH + SW feature panels of X per slab instead
// of two each.  That takes groups of workgroups that ARE super-tiles, so the whole ones come first, in row-major order, then
// those cut off by the last column, then the ones on the diagonal: with all of them in one row-major order the diagonal's
// shifted everything behind them, and a group straddled two super-tiles, 20 panels instead
// of 12.  L2 misses 1.22e8 -> 0.88e8 of 4.39e8 requests at 32768 x 14336 (12 panels for 64 reads are 0.82e8), 6.32 -> 5.99 ms;
// 8192 x 8192 598 -> 575 us.
__host__ __device__ __forceinline__ void tile_coords(int c, int nb, int SH, int SW, int& I, int& J) {
  const int rows = nb / SH, nsi = (nb + SH - 1) / SH;  // super-rows: whole ones, all
  const int cols = nb / SW, rest = nb % SW;
  // first super-column that lies right of the diagonal in all of super-row si
  auto first_right = [&](int si) { return (si * SH + SH - 1 + SW - 1) / SW; };
  for (int si = 0; si < rows; ++si) {
    const int f = first_right(si), n = f < cols ? (cols - f) * SH * SW : 0;
    if (c < n) {
      const int t = c % (SH * SW);
      I = si * SH + t / SW;
      J = (f + c / (SH * SW)) * SW + t % SW;
      return;
    }
    c -= n;
  }
  for (int si = 0; si < rows && rest > 0; ++si) {
    const int n = first_right(si) <= cols ? SH * rest : 0;
    if (c < n) {
      I = si * SH + c / rest;
      J = cols * SW + c % rest;
      return;
    }
    c -= n;
  }
  for (int si = 0; si < nsi; ++si) {
    // the columns from the diagonal up to the first super-column counted above (all of them in a cut-off super-row)
    const int f = first_right(si), c_hi = si < rows && (f < cols || (f == cols && rest > 0)) ? f * SW : nb;
    for (int i = si * SH; i < (si + 1) * SH && i < nb; ++i) {
      const int n = c_hi - i;
      if (c < n) {
        I = i;
        J = i + c;
        return;
      }
      c -= n > 0 ? n : 0;
    }
  }
  I = J = -1;
}
