// Fused demag kernels: F64 columns of 2^k points (registered at library load).
#include "demag_fused.hpp"
namespace {
struct Reg {
    Reg() { fused::register_mids<double, 8, 16, 32, 64>(); }
} reg;
}  // namespace
