// The large tiles' gated products (gemm_mfma_big.h), on the tile that the call names.
#include "gemm_mfma_big.h"

template <typename TO>
static int launch(const BigCall& c) {
#define FW_TILE(ROWS, COLUMNS, EACH) \
    if (c.slices <= 1 && c.rows == ROWS && c.columns == COLUMNS && c.each_cu == EACH) return launch_big<MB_SWIGLU, TO, COLUMNS / 64, ROWS / 64, EACH, false>(c);
    FW_BIG_WHOLE_TILES(FW_TILE)
#undef FW_TILE
    fw_set_error("gemm_mfma_big: no tile of %d x %d, %d on a compute unit, K in %d slices", c.rows, c.columns, c.each_cu, c.slices);
    return -1;
}

int fw_launch_big_gated(const BigCall& c) {
    if (c.out_dtype == FW_BF16_GEGLU) return launch<geglu_bf16_t>(c);
    return launch<bf16_t>(c);
}
