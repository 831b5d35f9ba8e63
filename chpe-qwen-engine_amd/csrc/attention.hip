// attention.hip -- the attention launches of the engine's steps (attention_kernels.hpp), positions from
// the device state.
#include "attention_kernels.hpp"

namespace chpe {

void launch_attention_partial(const AttnArgs& a, hipStream_t st) { launch_partial<false>(a, st); }
void launch_attention_combine(const AttnArgs& a, hipStream_t st) { launch_combine<false>(a, st); }

bool attention_supported(uint32_t H, uint32_t KV, uint32_t hd) {
  return KV > 0 && H % KV == 0 && ((hd == 128 && H / KV == 8) || (hd == 256 && H / KV == 4));
}

void launch_attention(const AttnArgs& a, hipStream_t st) {
  launch_attention_partial(a, st);
  launch_attention_combine(a, st);
}

}  // namespace chpe
