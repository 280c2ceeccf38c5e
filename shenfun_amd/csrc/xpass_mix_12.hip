#include "xpass_mix.h"

namespace sfa {

int xpass_mix_12(const XMixArgs& a, int64_t nb, hipStream_t s) { return xpass_mix_run<12>(a, nb, s); }

}  // namespace sfa
