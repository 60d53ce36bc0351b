// Instantiations of the register-coefficient kernel for one l_max and number
// of radial groups, MDX_BLOCK_LM and MDX_BLOCK_KG on the command line (build.py
// compiles this file once for each).
#include "soap_block_kernel.h"

#ifndef MDX_BLOCK_LM
#error "compile with -DMDX_BLOCK_LM=l_max -DMDX_BLOCK_KG=radial groups"
#endif

namespace mdx {
namespace {

// Shapes compiled in every form (float32 and float64 exps, with and without
// neighbour weights): the sizes this package's workloads use.  The others have
// float64 exps and five forms: unweighted float32 rows, and with weights that
// may be 1 (2-4 % slower than a form without them) rows, inner averages, inner
// averages of small structures and outer averages.
constexpr bool every_form(int lm, int kg, int ncr) {
    return (lm == 3 && kg == 1 && ncr == 1) || (lm == 6 && kg == 2 && ncr == 2) || (lm == 4 && kg == 2 && ncr == 3) ||
           (lm == 8 && kg == 2 && ncr == 3) || (lm == 9 && kg == 3 && ncr == 1);
}

template <int LM, int KG, int NCR>
constexpr BlockShape shape() {
    return {LM, KG, NCR, every_form(LM, KG, NCR), BlockPlan<LM, KG>::T, &launch_shape<LM, KG, NCR, every_form(LM, KG, NCR)>};
}

const BlockShape kShapes[] = {
    shape<MDX_BLOCK_LM, MDX_BLOCK_KG, 1>(),
    shape<MDX_BLOCK_LM, MDX_BLOCK_KG, 2>(),
#if MDX_BLOCK_KG > 1
    shape<MDX_BLOCK_LM, MDX_BLOCK_KG, 3>(),
#endif
#if MDX_BLOCK_KG > 2
    shape<MDX_BLOCK_LM, MDX_BLOCK_KG, 5>(),
#endif
};

} // namespace

#define MDX_NAME2(LM, KG) block_shapes_##LM##_##KG
#define MDX_NAME(LM, KG) MDX_NAME2(LM, KG)
std::pair<const BlockShape*, int> MDX_NAME(MDX_BLOCK_LM, MDX_BLOCK_KG)() {
    return {kShapes, static_cast<int>(sizeof(kShapes) / sizeof(kShapes[0]))};
}

} // namespace mdx
