// tbe_bag_walk.h — the order in which a kernel walks the rows of one bag.  Counts the
// rows that are left, never past the bag: a position counter that runs on past a bag of
// nearly 2^31 rows overflows, and its loop does not end.  Plain C++ besides, so that a
// host test can run it.
#ifndef TBE_BAG_WALK_H
#define TBE_BAG_WALK_H

#include <stdint.h>

#include <type_traits>

#if defined(__HIPCC__)
#define TBE_HD __host__ __device__ __forceinline__
#else
#define TBE_HD inline
#endif

namespace tbe {

// Steps of `step` rows in a pipeline of three stages over two register sets: indices of
// step s + 2, rows of step s + 1, sums of step s.  load(set, at, left) / issue(set, left)
// / consume(set, left): `left` rows remain from position `at` on (none: <= 0, at least
// -2 * step).  Stages past the bag are called too, so that every step issues the same
// loads.  L >= 1.
template <typename Load, typename Issue, typename Consume>
TBE_HD void walk_steps(int64_t at, int L, int step, Load load, Issue issue, Consume consume) {
  const std::integral_constant<int, 0> a{};
  const std::integral_constant<int, 1> b{};
  load(a, at, L);
  load(b, at + step, L - step);
  issue(a, L);
  for (int left = L;;) {
    load(a, at + 2 * step, left - 2 * step);
    issue(b, left - step);
    consume(a, left);
    at += step;
    left -= step;
    if (left <= 0) break;
    load(b, at + 2 * step, left - 2 * step);
    issue(a, left - step);
    consume(b, left);
    at += step;
    left -= step;
    if (left <= 0) break;
  }
}

// Chunks of up to `step` rows, one after another: body(position, rows).  left <= 0: none.
template <typename Body>
TBE_HD void walk_chunks(int64_t at, int left, int step, Body body) {
  for (; left > 0; left -= step, at += step) body(at, left < step ? left : step);
}

// Rows [first, first + rows) of a bag of len rows that wave `wave` of `waves` takes.
struct BagShare {
  int first, rows;
};
TBE_HD BagShare bag_share(int len, int wave, int waves) {
  const int per = len / waves + (len % waves != 0);
  const int first = wave * per < len ? wave * per : len;
  const int left = len - first;
  return {first, per < left ? per : left};
}

}  // namespace tbe

#endif  // TBE_BAG_WALK_H
