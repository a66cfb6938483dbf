// Fused demag kernels: F64 rows of 3 2^k and 5 2^k points (registered at library load).
#include "demag_fused.hpp"
namespace {
struct Reg {
    Reg() { fused::register_rows<double, 12, 24, 48, 96, 192, 384, 768, 10, 20, 40, 80, 160, 320, 640>(); }
} reg;
}  // namespace
