// Instantiations of the forward kernel for head dim 16 (fp16, bf16, and fp16 with a float8 e5m2 V).
#include "fa_fwd_kernel.hpp"
#include "kernel_table.hpp"

using namespace rsfa;

// (BN, NW, OCC) of the compiled tile shapes; overridable for tile sweeps.
// The softmax's VALU work bounds these head dims (four waves on a SIMD issue a
// v_fma every 3.9 cycles and a v_exp every 8.2; one alone 5.5 and 8.8), so four
// waves per SIMD: B=4 H=16 S=4096 causal 116 -> 108 us, B=32 H=8
// S=2048 209 -> 184.  Long non-causal rows take 128-key tiles with three (half the
// barriers: B=32 H=8 S=2048 179 us, float8 V B=16 S=1024 32.8 -> 28.1);
// causal ones lose at the wider diagonal (B=64 H=8 S=1024 65 us, 69).
#ifndef RSFA_D16_TILES
#define RSFA_D16_TILES(T, DTYPE) RSFA_TILE_ENTRIES(T, DTYPE, 16, 64, 4, 4), RSFA_TILE_NONCAUSAL(T, DTYPE, 16, 128, 4, 3)
#endif

RSFA_DEFINE_KERNEL_LIST(kernels_d16, RSFA_D16_TILES(TypeF16, 0), RSFA_D16_TILES(TypeBF16, 1),
                        RSFA_D16_TILES(TypeF16V8, 2))
