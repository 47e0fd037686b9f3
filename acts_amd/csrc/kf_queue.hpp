// kf_queue.hpp -- where in the track queue the tracks that may become
// loopers stand.
#pragma once

#include "kf_common.hpp"

namespace kf {

// The queue's sort puts the tracks that may become loopers first.  In one
// block they fill the first wavefronts, where loopers with different targets
// and step lengths take each other's steps too (a step of several in the
// field map 3.2 to 3.8 against 2.4 thousand x 4 cycles of one alone), which
// sets the length of a fit that is over before its loopers: forward kernel of
// 5 000 field-map tracks 4.6 -> 4.2 ms when they stand a wavefront apart,
// 100 000 7.1 -> 5.6, 200 000 7.2 -> 6.0.  A larger batch keeps the block: few
// wavefronts then stay behind in quarantine with their loopers while the
// others fit the rest (500 000: 6.7, spread 7.7 ms).  With fits in flight that
// is so from fewer tracks on, as the next fit's tracks fill the time; most with
// the layer navigator, whose tracks take longer beside loopers that do not:
// three fits in flight of 200 000 field-map tracks 21.1 ms spread, 18.6 in one
// block, of 250 000 24.6 and 21.5 (one alone 9.2 and 10.8, 9.6 and 10.8).
// There they stand four places apart from 2 batches of the resident lanes on,
// in a sixteenth of the wavefronts: 19.2 and 22.1 ms in flight, 10.1 and 10.0
// alone.
struct Spread {
  int32_t window;   // the first places, over which they are spread
  int32_t spacing;  // at most this many places apart
};
constexpr int32_t kWideSpacing = 64;  // a wavefront's places
constexpr int32_t kCloseSpacing = 4;
constexpr int64_t kSpreadBatch = 4, kWideBatchLayers = 2;  // in resident lanes
inline Spread spreadOf(int64_t n, int64_t lanes, bool layers) {
  if (n > kSpreadBatch * lanes) return Spread{1, 1};
  const bool wide = !layers || n <= kWideBatchLayers * lanes;
  return Spread{static_cast<int32_t>(n < lanes ? n : lanes), wide ? kWideSpacing : kCloseSpacing};
}

// Queue place of sorted place i: the nSeam first tracks up to s.spacing
// places apart in the window, the others between them.
KF_HD int32_t spreadPlace(int32_t i, int32_t nSeam, const Spread& s) {
  const int32_t fit = nSeam > 0 ? s.window / nSeam : 0;
  const int32_t spacing = fit < s.spacing ? fit : s.spacing;
  if (spacing <= 1) return i;
  const int32_t j = i - nSeam;
  if (j < 0) return i * spacing;
  if (j < nSeam * (spacing - 1)) return j / (spacing - 1) * spacing + 1 + j % (spacing - 1);
  return i;
}

}  // namespace kf
