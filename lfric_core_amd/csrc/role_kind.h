// Which compile-time table of column roles (colour_apply.h) a space's detected roles match.
#pragma once
#include "colour_apply.h"
#include "internal.h"
#include "kernels.h"

namespace lfric {
namespace {

// any pattern found in a caller's dofmap, beside the compile-time tables
struct RolesRuntime {
  static constexpr bool kStatic = false;
  Roles r;
  __device__ bool top(int i) const { return (r.top_mask >> i) & 1u; }
  __device__ int partner(int i) const { return r.partner[i]; }
};

// which compile-time role table (if any) a space's detected roles match
enum class RoleKind { None, W0K0, W0K1, W2K0, Runtime };
template <class R>
bool roles_match(const FunctionSpace &f) {
  for (int i = 0; i < f.ndf; ++i) {
    if (R::top(i) != static_cast<bool>((f.top_mask >> i) & 1u)) return false;
    if (R::partner(i) != f.partner[i]) return false;
  }
  return true;
}
inline RoleKind role_kind(const FunctionSpace &f) {
  if (f.ndf == 8 && roles_match<RolesW0K0>(f)) return RoleKind::W0K0;
  if (f.ndf == 27 && roles_match<RolesW0K1>(f)) return RoleKind::W0K1;
  if (f.ndf == 6 && roles_match<RolesW2K0>(f)) return RoleKind::W2K0;
  if (roles_match<RolesNone>(f)) return RoleKind::None;
  return RoleKind::Runtime;
}

}  // namespace
}  // namespace lfric
