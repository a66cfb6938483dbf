// Fused demag kernels: F64 columns of 5 2^k points (registered at library load).
#include "demag_fused.hpp"
namespace {
struct Reg {
    Reg() { fused::register_mids<double, 10, 20, 40, 80, 160, 320, 640>(); }
} reg;
}  // namespace
