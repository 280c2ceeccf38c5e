#include "xpass_mix.h"

namespace sfa {

int xpass_mix_8(const XMixArgs& a, int64_t nb, hipStream_t s) { return xpass_mix_run<8>(a, nb, s); }

}  // namespace sfa
