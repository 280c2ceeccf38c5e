#include "mix_line.h"

namespace sfa {

int mix_run_fft(int, bool inv, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    return inv ? mix_run<OP_C2C, true, true>(a, grid, block, lds, stream) : mix_run<OP_C2C, false, true>(a, grid, block, lds, stream);
}

}  // namespace sfa
