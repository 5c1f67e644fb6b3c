// Instantiations of the forward kernel for head dim 32 (fp16, bf16, and fp16 with a float8 e5m2 V).
#include "fa_fwd_keysplit.hpp"
#include "kernel_table.hpp"

using namespace rsfa;

// (BN, NW, OCC) of the compiled tile shapes; overridable for tile sweeps.
// The softmax's VALU work bounds these head dims (four waves on a SIMD issue a
// v_fma every 3.9 cycles and a v_exp every 8.2; one alone 5.5 and 8.8), so four
// waves per SIMD: B=4 H=16 S=4096 causal 131 -> 116 us, B=64 H=8 S=2048 causal
// 286 -> 241, B=32 H=16 S=333 25.7 -> 23.1.  Long non-causal rows take 128-key tiles with three (half the
// barriers: B=32 H=8 S=2048 229 -> 211 us, 220 with 64 keys; float8 V B=16
// S=1024 34.8 -> 29.9, 30.6);
// causal ones lose at the wider diagonal (B=4 H=16 S=4096 130 us).
#ifndef RSFA_D32_TILES
#define RSFA_D32_TILES(T, DTYPE) RSFA_TILE_ENTRIES(T, DTYPE, 32, 64, 4, 4), RSFA_TILE_NONCAUSAL(T, DTYPE, 32, 128, 4, 3)
#endif

#define RSFA_D32_KS(T, DTYPE) RSFA_KEYSPLIT_ENTRIES(T, DTYPE, 32, 128, 64, 64, 4)

RSFA_DEFINE_KERNEL_LIST(kernels_d32, RSFA_D32_TILES(TypeF16, 0), RSFA_D32_TILES(TypeBF16, 1),
                        RSFA_D32_TILES(TypeF16V8, 2), RSFA_D32_KS(TypeF16, 0), RSFA_D32_KS(TypeBF16, 1))
