// Fused demag kernels: F64 columns of 3 2^k points (registered at library load).
#include "demag_fused.hpp"
namespace {
struct Reg {
    Reg() { fused::register_mids<double, 12, 24, 48, 96, 192, 384, 768>(); }
} reg;
}  // namespace
