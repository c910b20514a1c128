// Instantiates the NTT pass shapes beyond the planner's static choice for
// u64 words, lazy and strict.
#include "ntt_kernels.hpp"

namespace cbw {
namespace ntt_detail {
void register_alt_u64() {
    add_alt_u64<kLazy>();
    add_alt_u64<kStrict>();
}
}  // namespace ntt_detail
}  // namespace cbw
