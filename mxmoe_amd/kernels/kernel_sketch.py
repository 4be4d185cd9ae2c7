"""Source templates of the generated gfx950 kernels (role of the reference's mxmoe/kernels/kernel_sketch.py).

The reference expands a 400-line CUDA string per kernel.  Here the device code lives in the header tile library
(csrc/include/mxmoe_tiles.hpp, mxmoe_wo_tiles.hpp) and the fused kernel + host launcher are a variadic template
(csrc/include/mxmoe_launch.hpp), so a generated translation unit only names the tile types of its branches.
"""
from string import Template

KERNEL_DEFINITION_TEMPLATE = Template("""// generated by mxmoe_amd.kernels.compose_kernel — do not edit
// ${Comment}
#include "mxmoe_launch.hpp"

namespace mxmoe {
namespace {
struct Register_${KernelName} {
  Register_${KernelName}() {
    register_fused<${Tiles}>("${KernelName}", ${Policy}${Hint});
  }
};
static Register_${KernelName} register_${KernelName};
}  // namespace
}  // namespace mxmoe
""")

# One kernel of a library whose kernels are spread over several translation units: the unit only defines the registration function,
# and DEFAULT_ORDER_TEMPLATE calls them in registry order (static initialisers of different units have no order of their own).
KERNEL_DEFERRED_TEMPLATE = Template("""// generated by mxmoe_amd.kernels.compose_kernel — do not edit
// ${Comment}
#include "mxmoe_launch.hpp"

namespace mxmoe {
int register_${KernelName}() { return ${Register}<${Tiles}>("${KernelName}", ${Policy}${Hint}); }
}  // namespace mxmoe
""")

DEFAULT_ORDER_TEMPLATE = Template("""// generated by mxmoe_amd.kernels.compose_kernel — do not edit
// Registers the kernels of this library in registry order.
namespace mxmoe {
${Decls}
namespace {
struct RegisterAll {
  RegisterAll() {
${Calls}
  }
};
static RegisterAll register_all;
}  // namespace
}  // namespace mxmoe
""")

KERNEL_DECLARATION_TEMPLATE = Template("""// generated by mxmoe_amd.kernels.compose_kernel — do not edit
// Kernels of this library, in registry order:
${Signatures}
""")

ABI_TU = """// generated by mxmoe_amd.kernels.compose_kernel — do not edit
// The C-ABI entry points of this generated library (same symbols as libmxmoe_amd.so, own registry).
#include "mxmoe_abi_impl.hpp"
"""
