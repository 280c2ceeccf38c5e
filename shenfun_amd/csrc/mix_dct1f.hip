#include "mix_line.h"

namespace sfa {

int mix_run_dct1f(bool cplx, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    if (a.K2)
        return cplx ? mix_run<OP_DCT1F, false, true, true>(a, grid, block, lds, stream)
                    : mix_run<OP_DCT1F, false, false, true>(a, grid, block, lds, stream);
    return cplx ? mix_run<OP_DCT1F, false, true, false>(a, grid, block, lds, stream)
                : mix_run<OP_DCT1F, false, false, false>(a, grid, block, lds, stream);
}

}  // namespace sfa
