// Fused demag kernels: F64 rows of 2^k points (registered at library load).
#include "demag_fused.hpp"
namespace {
struct Reg {
    Reg() { fused::register_rows<double, 8, 16, 32, 64, 128, 256, 512, 1024>(); }
} reg;
}  // namespace
