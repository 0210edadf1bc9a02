// feat3amd_check.hpp -- the word in which a set-up kernel leaves the verdict of a check.
#pragma once

#include <cstdint>

namespace feat3amd_detail {

// The word starts at 0.  The checking kernel adds kCheckRan once and kCheckBad for every place
// that fails; only kCheckRan alone passes.  A word that the kernel never wrote, or that the
// host read before it was there, therefore fails, and the plan takes its general form.
constexpr uint32_t kCheckRan = 0x5EED0000u;
constexpr uint32_t kCheckBad = 1u;

constexpr bool check_passed(uint32_t word) { return word == kCheckRan; }

} // namespace feat3amd_detail
