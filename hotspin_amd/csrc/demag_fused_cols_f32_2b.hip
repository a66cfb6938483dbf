// Fused demag kernels: F32 columns of 2^k points (registered at library load).
#include "demag_fused.hpp"
namespace {
struct Reg {
    Reg() { fused::register_mids<float, 128, 256, 512, 1024>(); }
} reg;
}  // namespace
