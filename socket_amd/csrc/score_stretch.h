// Where the persistent scorer's stretches of the row space begin (score_deal.h).  Plain arithmetic: it compiles for the host too.
#pragma once
#include <stdint.h>

// Units [start, start + size) of `total` for stretch `group` of `groups`: start is total * group / groups rounded down, so
// that the remainder is spread evenly over the groups and stretches end where rows do wherever the two divide.  In 32 bits
// (group < groups <= 65535): total * g / n = each * g + more * g / n, with each = total / n and more = total % n.
// (The remainder given to the first groups instead, a unit each: no faster where a workgroup has no more than a unit, and
// groups follow one another by XCD, so it left whole XCDs idle or with twice the work, and stretches over the ends of rows,
// two tables where one would do.  us, that / this: 8 kv heads of 4, 60 tables x 1024, capacity 131072, 4000 cached tokens 14.8 / 14.7,
// 12000 26.0 / 14.7, 40000 26.8 / 16.0.)
struct ScoreStretch {
  uint32_t start, size;
};

constexpr ScoreStretch score_stretch(uint32_t total, uint32_t group, uint32_t groups) {
  const uint32_t each = total / groups, more = total - each * groups;
  const uint32_t before = more * group / groups, rest = more * group - before * groups;
  return {each * group + before, each + (rest + more >= groups ? 1u : 0u)};
}
