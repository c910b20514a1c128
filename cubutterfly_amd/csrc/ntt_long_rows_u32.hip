// Instantiates the one-pass NTT kernels of 2^13- and 2^14-point rows for u32
// words, lazy and strict.
#include "ntt_kernels.hpp"

namespace cbw {
namespace ntt_detail {
void register_long_rows_u32() {
    add_long_rows<std::uint32_t, kLazy>();
    add_long_rows<std::uint32_t, kStrict>();
}
}  // namespace ntt_detail
}  // namespace cbw
