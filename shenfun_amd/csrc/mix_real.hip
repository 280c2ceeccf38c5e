#include "mix_line.h"

namespace sfa {

int mix_run_real(int op, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    switch (op) {
        case OP_R2C: return mix_run<OP_R2C, false, false>(a, grid, block, lds, stream);
        case OP_C2R: return mix_run<OP_C2R, true, true>(a, grid, block, lds, stream);
        case OP_R2CF: return mix_run<OP_R2CF, false, false>(a, grid, block, lds, stream);
        default: return mix_run<OP_C2RF, true, false>(a, grid, block, lds, stream);
    }
}

}  // namespace sfa
