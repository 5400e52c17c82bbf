// wavesum.hpp -- sums of several values over a wave at once.
#pragma once
#include <hip/hip_runtime.h>

namespace spined {

// Sums of acc[0..NQ) over the 64 lanes.  At each of the six levels a lane
// hands half of its values to its partner and keeps the other half, so NQ
// values take about NQ + 4 exchanges instead of 6 NQ (25 values: 28 for 150).
// Level by level the same pairs are added as in the tree
//   for (off = 32; off > 0; off >>= 1) v += shfl_down(v, off),
// so each sum has the bits of that tree.  Returns this lane's sum; `index` is
// the value it belongs to, -1 where the lane holds none.
template <int NQ>
__device__ inline double wave_sums(const double (&acc)[NQ], int lane, int &index) {
  if constexpr (NQ == 1) {
    double v = acc[0];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    index = lane == 0 ? 0 : -1;
    return v;
  } else {
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) v[q] = acc[q];
    int first = 0, left = NQ; // this lane's values: first .. first + left
    int n = NQ;               // slots in use, a constant at each unrolled level
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int h = (n + 1) / 2;
      const bool up = (lane & off) != 0;
#pragma unroll
      for (int i = 0; i < h; ++i) {
        const double hi = h + i < n ? v[h + i] : 0.0;
        const double got = __shfl_xor(up ? v[i] : hi, off, 64);
        v[i] = (up ? hi : v[i]) + got;
      }
      first += up ? h : 0;
      left = up ? left - h : (left < h ? left : h);
      n = h;
    }
    index = left > 0 ? first : -1;
    return v[0];
  }
}

} // namespace spined
