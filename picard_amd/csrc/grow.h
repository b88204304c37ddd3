// grow.h -- an array that grows with what it holds: the new one is there before the old one goes,
// so that a failure leaves the old one as it was.
#pragma once
#include <cstdint>

namespace picard {

// Room for `want` entries, `per` elements each, in *p (*cap entries so far).  alloc(&q, elements) and
// give_back(old) return 0 or an error, which is passed on; give_back is called before *p changes.
template <typename T, typename Alloc, typename GiveBack>
int grow_array(T **p, int64_t *cap, int64_t want, int64_t per, const Alloc &alloc, const GiveBack &give_back) {
  if (want <= *cap) return 0;
  const int64_t n = want + want / 2;
  T *q = nullptr;
  if (const int rc = alloc(&q, per * n)) return rc;
  if (const int rc = give_back(*p)) return rc;
  *p = q;
  *cap = n;
  return 0;
}

}  // namespace picard
