// step_f32_exact5.hip -- the fast step kernels of the exact solver for gamma =
// 5/3 (step_f32_kernel.hpp).
#define AST_STEP_F32_KERNELS
#include "step_f32_kernel.hpp"

namespace ast {
namespace f32 {
template int step_launch<kExact5>(const StepArgs&);
}  // namespace f32
}  // namespace ast
