// The device headers as strings: the builtins are prepended to every hiprtc translation unit.
#include "codegen.hpp"

namespace ocannl {
const char* builtins_hip_source() {
  static const char text[] =
#include "builtins_hip.inc"
      ;
  return text;
}
const char* contract_any_source() {
  static const char text[] =
#include "contract_any.inc"
      ;
  return text;
}
}  // namespace ocannl
