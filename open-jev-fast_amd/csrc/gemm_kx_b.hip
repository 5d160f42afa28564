// K-interleaved tiles, part b: the instantiations of gemm_kx.h are spread over three translation units so that they
// compile side by side. Registered in gemm.hip's tile table; BN x BM = 16 FW x 16 (4 FX + XE).
#include "gemm_kx.h"

namespace ojx {
template GemmFn kx_pick<9, 2, 1, 2>(int, bool);  // 144 x 144
template GemmFn kx_pick<16, 2, 0, 2>(int, bool);  // 256 x 128: one head per tile
template GemmFn kx_pick<16, 1, 0, 2>(int, bool);  // 256 x 64
template GemmFn kx_pick<10, 2, 0, 2>(int, bool);  // 160 x 128
template GemmFn kx_pick<8, 2, 2, 2>(int, bool);  // 128 x 160
template GemmFn kx_pick<8, 3, 2, 2>(int, bool);  // 128 x 224
template GemmFn kx_pick<9, 3, 2, 2>(int, bool);  // 144 x 224
}  // namespace ojx
