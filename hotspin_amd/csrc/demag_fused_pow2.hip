// Fused demag kernels for lengths 2^k (registered at library load).
#include "demag_fused.hpp"
namespace {
template <typename T>
void reg_all() {
    fused::register_len<T, 8>(); fused::register_len<T, 16>(); fused::register_len<T, 32>();
    fused::register_len<T, 64>(); fused::register_len<T, 128>(); fused::register_len<T, 256>();
    fused::register_len<T, 512>(); fused::register_len<T, 1024>();
}
struct Reg {
    Reg() {
        reg_all<float>();
        reg_all<double>();
    }
} reg;
}  // namespace
