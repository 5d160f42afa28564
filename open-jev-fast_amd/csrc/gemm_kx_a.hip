// K-interleaved tiles, part a: the instantiations of gemm_kx.h are spread over three translation units so that they
// compile side by side. Registered in gemm.hip's tile table; BN x BM = 16 FW x 16 (4 FX + XE).
#include "gemm_kx.h"

namespace ojx {
template GemmFn kx_pick<9, 4, 2, 2>(int, bool);  // 144 x 288
template GemmFn kx_pick<8, 4, 2, 2>(int, bool);  // 128 x 288
template GemmFn kx_pick<8, 4, 0, 2>(int, bool);  // 128 x 256
template GemmFn kx_pick<10, 4, 0, 2>(int, bool);  // 160 x 256
template GemmFn kx_pick<9, 3, 0, 2>(int, bool);  // 144 x 192
}  // namespace ojx
