// Fused demag kernels for lengths 3 * 2^k and 5 * 2^k (registered at library load).
#include "demag_fused.hpp"
namespace {
template <typename T>
void reg_all() {
    fused::register_len<T, 12>(); fused::register_len<T, 24>(); fused::register_len<T, 48>();
    fused::register_len<T, 96>(); fused::register_len<T, 192>(); fused::register_len<T, 384>();
    fused::register_len<T, 768>();
    fused::register_len<T, 10>(); fused::register_len<T, 20>(); fused::register_len<T, 40>();
    fused::register_len<T, 80>(); fused::register_len<T, 160>(); fused::register_len<T, 320>();
    fused::register_len<T, 640>();
}
struct Reg {
    Reg() {
        reg_all<float>();
        reg_all<double>();
    }
} reg;
}  // namespace
