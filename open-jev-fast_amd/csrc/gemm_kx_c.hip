// K-interleaved tiles, part c: the instantiations of gemm_kx.h are spread over three translation units so that they
// compile side by side. Registered in gemm.hip's tile table; BN x BM = 16 FW x 16 (4 FX + XE).
#include "gemm_kx.h"

namespace ojx {
template GemmFn kx_pick<9, 1, 0, 2>(int, bool);  // 144 x 64
template GemmFn kx_pick<9, 2, 0, 2>(int, bool);  // 144 x 128
template GemmFn kx_pick<8, 2, 0, 2>(int, bool);  // 128 x 128
template GemmFn kx_pick<8, 1, 0, 2>(int, bool);  // 128 x 64
template GemmFn kx_pick<8, 1, 0, 4>(int, bool);  // 128 x 64, 4 stages ahead
template GemmFn kx_pick<8, 1, 2, 2>(int, bool);  // 128 x 96
}  // namespace ojx
