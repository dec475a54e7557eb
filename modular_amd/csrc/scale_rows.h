// The row of the weight scales (one per 128 weight rows) that serves the columns of C from n on.
#pragma once

namespace maxfp8 {

// n may lie past the last column: a tile reaches up to its own width past N, and a wave of it whose columns all lie there stores nothing but reads
// its scale like the others.  It takes the last row: the row behind that is not the operand's, and with scales that end where their
// allocation does, reading it faults (128 matrices of one scale each under 256 columns wide tiles: the 129th of 128 floats).
constexpr int weight_scale_row(int n, int N) {
  const int row = n / 128, last = (N - 1) / 128;
  return row < last ? row : last;
}

}  // namespace maxfp8
