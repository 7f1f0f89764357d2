// The products on large tiles that are asked for by shape: the plan of the tile, K cut over workgroups, the experts' grouped product, and the tile named
// by the caller. The kernel is gemm_mfma_big.h.
#include <math.h>

#include "gemm_mfma_big.h"

// The grouped product of fw_grouped_gemm, for K a multiple of 32 and a of less than 4 GB. Bound by the experts' weights from memory (600 MB for both products
// of 32 experts of 1,536 features: 127 us), by tiles that an expert's last places fill partly and by rounds of them that the chip is not full with: the tile
// follows from how many places an expert has in the mean. us, tiles of 128 x 256 alone / chosen, gated and down: 32 experts of 1,536 features over 2,048, four
// a row, 2,048 rows 160 / 145 and 93 / 77, 1,111 rows 129 / 105 and 65 / 49, 600 rows 103 / 97 and 50 / 45; 16 of 1,024 over 4,096, two a row, 2,048 rows 123 / 88 and
// 66 / 55; 64 of 768 over 1,024, six a row, 3,000 rows 109 / 91 and 60 / 50. All tiles give the same bits.
bool fw_grouped_big_takes(int a_rows, int N, int K) { return K % BK == 0 && K <= BK_MOST && N <= BN_MOST && 2ll * a_rows * K <= 0xffff0000ll; }

// What a tile takes, us: start + rounds * round + tiles / 256 * tile + K / 1,024 * (rounds * walk + tiles / 256 * fill) + MB of all experts' weights * memory,
// rounds those of the tiles over 256 compute units (512 places where two workgroups share one). Fitted to 60 shapes a form (8 to 128 experts, 200 to
// 4,000 rows) to 5 to 10 % (mean square); so chosen they take 1.5 (gated) and 2.4 % (down) more than with the fastest tile each, and 9 and 12 % less than with one tile.
struct GroupedTime {
    int rows, columns, each_cu;
    float start, round, tile, walk, fill, memory;
};
static const GroupedTime grouped_times[2][7] = {
    {{64, 128, 2, 0.00f, 1.69f, 0.31f, 1.81f, 4.66f, 0.10f},
     {128, 128, 2, 0.00f, 4.18f, 0.00f, 3.18f, 6.26f, 0.07f},
     {128, 192, 1, 0.00f, 0.00f, 4.39f, 5.27f, 6.19f, 0.09f},
     {128, 256, 1, 0.00f, 5.89f, 0.00f, 7.40f, 4.88f, 0.09f},
     {192, 192, 1, 0.00f, 0.00f, 5.07f, 7.64f, 7.53f, 0.06f},
     {192, 256, 1, 0.00f, 7.53f, 0.00f, 10.33f, 7.58f, 0.05f},
     {256, 256, 1, 0.00f, 10.03f, 0.00f, 12.41f, 5.93f, 0.06f}},
    {{64, 128, 2, 1.16f, 0.00f, 0.96f, 5.69f, 1.95f, 0.11f},
     {128, 128, 2, 4.24f, 2.27f, 0.00f, 3.57f, 5.23f, 0.09f},
     {128, 192, 1, 4.36f, 4.89f, 0.00f, 8.30f, 1.44f, 0.09f},
     {128, 256, 1, 0.32f, 5.96f, 0.38f, 7.08f, 3.95f, 0.11f},
     {192, 192, 1, 0.69f, 7.95f, 0.00f, 10.28f, 1.73f, 0.07f},
     {192, 256, 1, 11.21f, 5.31f, 0.00f, 5.18f, 11.60f, 0.07f},
     {256, 256, 1, 10.72f, 7.17f, 0.00f, 8.36f, 13.75f, 0.04f}}};

// Tiles of `rows` places that experts of `mean` places in the mean have, their numbers spread as independent choices spread them (the device alone knows them):
// the sum over j of the chance that an expert has more than j * rows.
static double expected_tiles(double mean, int rows) {
    double tiles = 0.0;
    for (int j = 0;; ++j) {
        const double chance = 0.5 * erfc((j * (double)rows + 0.5 - mean) / sqrt(2.0 * mean));
        if (chance < 1e-3) return tiles;
        tiles += chance;
    }
}

static const GroupedTime& grouped_plan(int gated, int places, int experts, int N, int K, bool tall) {
    const GroupedTime* best = nullptr;
    double least = 0.0;
    for (const GroupedTime& t : grouped_times[gated]) {
        if (t.rows > 128 && !tall) continue;
        const double tiles = expected_tiles((double)places / experts, t.rows) * experts * fw_ceil_div(N, gated ? t.columns / 2 : t.columns), share = tiles / 256.0;
        const double rounds = ceil(tiles / (256.0 * t.each_cu)), k = K / 1024.0;
        const double time = t.start + rounds * t.round + share * t.tile + k * (rounds * t.walk + share * t.fill) + 2e-6 * experts * (gated ? 2.0 : 1.0) * N * K * t.memory;
        if (!best || time < least) {
            best = &t;
            least = time;
        }
    }
    return *best;
}

// The tile of a grouped product that goes straight to LDS.
extern "C" int fw_grouped_gemm_tile(int gated, int places, int experts, int N, int K, int tall, int* rows, int* columns) {
    FW_REQUIRE(places >= 1 && experts >= 1 && N >= 1 && K >= 1, "grouped_gemm_tile: bad sizes places=%d experts=%d N=%d K=%d", places, experts, N, K);
    const GroupedTime& plan = grouped_plan(gated ? 1 : 0, places, experts, N, K, tall != 0);
    *rows = plan.rows;
    *columns = plan.columns;
    return 0;
}

// `tiled`: w in operand tiles; `tall`: tiles of more than 128 places are worth a look (fw_grouped_gemm_large_fits)
int fw_launch_grouped_big(const void* a, const int32_t* place_row, const void* w, bool tiled, const int32_t* expert_begin, void* out, int gated, int places,
                          int experts, int N, int K, bool tall, hipStream_t stream) {
    const BigGroups groups = {place_row, expert_begin, experts, tiled};
    const GroupedTime& plan = grouped_plan(gated, places, experts, N, K, tall);
    const int tiles_m = places / plan.rows + (experts < places ? experts : places);       // at most: every expert's last tile may not be full
    // (what the product through registers, whose tiles have half the features, would refuse is refused here too)
    FW_REQUIRE((long long)(places / 128 + (experts < places ? experts : places)) * fw_ceil_div(N, gated ? BT / 4 : BT / 2) < (1ll << 30), "grouped_gemm: too many tiles");
    FW_REQUIRE((long long)tiles_m * fw_ceil_div(N, gated ? plan.columns / 2 : plan.columns) < (1ll << 30), "grouped_gemm: too many tiles");
#define FW_GROUPED_TILE(ROWS, COLUMNS, EACH)                                                                                                                   \
    if (plan.rows == ROWS && plan.columns == COLUMNS && plan.each_cu == EACH)                                                                                  \
        return gated ? launch_tiles<MB_SWIGLU, bf16_t, COLUMNS / 64, ROWS / 64, true, false, EACH>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream) \
                     : launch_tiles<MB_STORE, float, COLUMNS / 64, ROWS / 64, true, false, EACH>(a, w, nullptr, out, places, N, K, tiles_m, groups, stream)
    FW_GROUPED_TILE(64, 128, 2);
    FW_GROUPED_TILE(128, 128, 2);
    FW_GROUPED_TILE(128, 192, 1);
    FW_GROUPED_TILE(128, 256, 1);
    FW_GROUPED_TILE(192, 192, 1);
    FW_GROUPED_TILE(192, 256, 1);
    FW_GROUPED_TILE(256, 256, 1);
#undef FW_GROUPED_TILE
    fw_set_error("grouped_gemm: no tile of %d x %d", plan.rows, plan.columns);
    return -1;
}

// The tile a storing or accumulating product is cut into: 256 or 128 rows by 256 or 192 columns,
// whichever takes the least time by this count: rounds of tiles over the chip's 256 compute units
// times the tile's area, a tile of 128 rows counting a quarter more than its area (it moves more
// bytes per flop). Gated products (SwiGLU) keep 256 x 256. (2,048 x 3,072 x 2,048: storing 50.9 -> 35.6 us with tiles of
// 128 x 192. Accumulating ones asked for each old value behind the store of the one before it and lost with twice the tiles; asked
// for a column of the tile at a time they gain as well.)
struct BigPlan {
    int rows, columns, tiles;
};
static BigPlan big_plan(int mode, int M, int N) {
    if (mode == MB_SWIGLU) return {BT, BT / 2, fw_ceil_div(M, BT) * fw_ceil_div(N, BT / 2)};
    BigPlan best = {0, 0, 0};
    long long best_cost = 0;
    for (int rows = BT; rows >= BT / 2; rows /= 2)
        for (int columns = BT; columns >= 192; columns -= 64) {
            const long long tiles = (long long)fw_ceil_div(M, rows) * fw_ceil_div(N, columns);
            const long long cost = fw_ceil_div(tiles, 256) * (rows / 32) * (columns / 32) * (rows == BT ? 4 : 5);
            if (best.tiles == 0 || cost < best_cost) {
                best = {rows, columns, (int)(tiles < (1ll << 30) ? tiles : (1ll << 30))};
                best_cost = cost;
            }
        }
    return best;
}

// How many tiles the kernel cuts a shape into, by the tile it will choose, and that tile's edges (the caller works out from them
// whether that fills the chip); 0 if the kernel does not take the shape (K must be a multiple of 32).
extern "C" int fw_gemm_mfma_big_plan(int mode, int M, int N, int K, int* rows, int* columns) {
    if (K <= 0 || K % BK || K > BK_MOST || M < 1 || N < 1 || N > BN_MOST) return 0;
    const BigPlan plan = big_plan(mode, M, N);
    if (rows) *rows = plan.rows;
    if (columns) *columns = plan.columns;
    return plan.tiles;
}

static int launch(int mode, const BigCall& call) {
    return mode == MB_SWIGLU ? fw_launch_big_gated(call) : mode == MB_ACCUMULATE ? fw_launch_big_add(call) : fw_launch_big_store(call);
}

// What every product on large tiles asks of its operands and outputs.
static int check_operands(const void* a, const void* w, const float* bias, int out_dtype, int mode, int M, int N, int K) {
    FW_REQUIRE(M >= 1 && N > 0 && K > 0 && K % BK == 0, "gemm_mfma_big: K (%d) must be a positive multiple of %d; M=%d N=%d", K, BK, M, N);
    FW_REQUIRE(mode >= 0 && mode <= 2, "gemm_mfma_big: unknown mode %d", mode);
    FW_REQUIRE(mode != MB_ACCUMULATE || out_dtype == FW_F32, "gemm_mfma_big: accumulation needs a float32 destination");
    FW_REQUIRE(mode != MB_SWIGLU || ((out_dtype == FW_BF16 || out_dtype == FW_BF16_GEGLU) && bias == nullptr), "gemm_mfma_big: SwiGLU stores bfloat16 and takes no bias");
    FW_REQUIRE(out_dtype == FW_F32 || out_dtype == FW_BF16 || (out_dtype == FW_BF16_GELU && mode == MB_STORE) || (out_dtype == FW_BF16_GEGLU && mode == MB_SWIGLU), "gemm_mfma_big: unknown out dtype %d", out_dtype);
    FW_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_mfma_big: operands must be 16-byte aligned");
    return 0;
}

// Same contract as fw_gemm_mfma.
extern "C" int fw_gemm_mfma_big(const void* a, const void* w, const float* bias, void* out, int out_dtype, int mode,
                                int M, int N, int K, void* stream) {
    if (check_operands(a, w, bias, out_dtype, mode, M, N, K)) return -1;
    FW_REQUIRE((long long)fw_ceil_div(M, BT / 2) * fw_ceil_div(N, BT / 2) < (1ll << 30), "gemm_mfma_big: too many tiles");
    // rows too long for a lane's 32-bit places (8 MB of an operand, 4 MB of the output) go through registers, with 64-bit addresses
    if (K > BK_MOST || N > BN_MOST) return fw_gemm_mfma(a, w, bias, out, out_dtype, mode, M, N, K, stream);
    const BigPlan plan = big_plan(mode, M, N);
    if (launch(mode, {a, w, bias, out, out_dtype, M, N, K, plan.rows, mode == MB_SWIGLU ? BT : plan.columns, 1, 1, K, nullptr, nullptr, (hipStream_t)stream})) return -1;
    FW_LAUNCH_CHECK("gemm_mfma_big");
    return 0;
}

// ----- K cut into slices, for products with at most half as many tiles as compute units and a long K --------
// A tile of 128 x 256 moves 48 bytes a clock of full MFMA rate through a compute unit's memory path, one of 128 x 128 all of its 64: two or three slices of K on
// the larger tiles pay for their meeting (about 12 us: 128 KB a workgroup out past the dies' caches and back) where K is long. us, cut / 128 x 128 with
// K dealt to the waves: storing 1,111 x 2,048 x 8,192 49.6 / 60.3, adding 2,048 x 2,048 x 8,192 72.2 / 70.5 alone and 8 us less of it in a prompt's step
// (4,863 against 4,995 for 16 layers), storing 1,024 x 2,560 x 6,368 51.2 / 73 (whole large tiles). With four slices the sum at the end costs more than it
// gives (adding 801 x 2,048 x 7,168 40.6 against 38.7 on 128 x 64), and so do slices of less than 512 k (2,048 x 1,024 x 1,024 21.2 / 12.2).
struct BigSplitPlan {
    int tiles, slices, k_each;
    size_t workspace_bytes;
};
static BigSplitPlan big_split_plan(int M, int N, int K) {
    BigSplitPlan plan = {0, 0, 0, 0};
    const long long tiles = (long long)fw_ceil_div(M, BT / 2) * fw_ceil_div(N, BT);
    if (tiles > 128) return plan;
    int slices = (int)(256 / tiles);                    // at most a workgroup a compute unit
    slices = slices > 3 ? 3 : slices;                   // the last workgroup of a tile adds them one after the other
    const int most = K / 512;
    slices = slices > most ? most : slices;
    if (slices < 2) return plan;
    plan.tiles = (int)tiles;
    plan.k_each = fw_ceil_div(fw_ceil_div(K, slices), 64) * 64;
    plan.slices = fw_ceil_div(K, plan.k_each);
    plan.workspace_bytes = (size_t)plan.slices * plan.tiles * (BT / 2) * BT * sizeof(float);
    return plan;
}

// What fw_gemm_mfma_big_split needs for a shape: its slices of K (0: it does not take the shape), bytes of float32 workspace and the number of
// int32 counters (zero before the first call; left zero).
extern "C" int fw_gemm_mfma_big_split_plan(int mode, int M, int N, int K, int* slices, size_t* workspace_bytes, int* counters) {
    FW_REQUIRE(M >= 1 && N > 0 && K > 0 && mode >= 0 && mode <= 2, "gemm_mfma_big_split: M %d N %d K %d mode %d", M, N, K, mode);
    BigSplitPlan plan = {0, 0, 0, 0};
    if (mode != MB_SWIGLU && K % BK == 0 && K <= BK_MOST && N <= BN_MOST) plan = big_split_plan(M, N, K);
    *slices = plan.slices;
    *workspace_bytes = plan.workspace_bytes;
    *counters = plan.tiles;
    return 0;
}

// fw_gemm_mfma's contract for modes 0 and 1, with K cut into slices as fw_gemm_mfma_big_split_plan says, on tiles of 128 x 256. Calls that overlap on one
// device must not share counters or workspace.
extern "C" int fw_gemm_mfma_big_split(const void* a, const void* w, const float* bias, void* out, int out_dtype, int mode, int M, int N, int K,
                                      void* workspace, size_t workspace_bytes, int* counters, int counters_len, void* stream) {
    int slices = 0, need_counters = 0;
    size_t need_bytes = 0;
    if (fw_gemm_mfma_big_split_plan(mode, M, N, K, &slices, &need_bytes, &need_counters)) return -1;
    FW_REQUIRE(slices > 1, "gemm_mfma_big_split: this shape (M %d N %d K %d mode %d) is not cut", M, N, K, mode);
    FW_REQUIRE(mode != MB_ACCUMULATE || out_dtype == FW_F32, "gemm_mfma_big_split: accumulation needs a float32 destination");
    FW_REQUIRE(out_dtype == FW_F32 || out_dtype == FW_BF16 || (out_dtype == FW_BF16_GELU && mode == MB_STORE), "gemm_mfma_big_split: unknown out dtype %d", out_dtype);
    FW_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_mfma_big_split: operands must be 16-byte aligned");
    FW_REQUIRE(workspace != nullptr && workspace_bytes >= need_bytes && counters != nullptr && counters_len >= need_counters && (uintptr_t)workspace % 16 == 0,
               "gemm_mfma_big_split: this shape needs %zu bytes of workspace and %d counters", need_bytes, need_counters);
    const BigSplitPlan plan = big_split_plan(M, N, K);
    if (launch(mode, {a, w, bias, out, out_dtype, M, N, K, BT / 2, BT, 1, plan.slices, plan.k_each, (float*)workspace, counters, (hipStream_t)stream})) return -1;
    FW_LAUNCH_CHECK("gemm_mfma_big_split");
    return 0;
}

// ----- the tile named by the caller --------
// 64 x 128 and 128 x 128 tiles with K cut into up to eight slices serve the products of a few hundred rows whose tiles would leave compute units idle: adding
// 801 x 2,048 x 7,168 43.3 -> 36.1 us in two slices of 128 x 128 (the waves splitting K before), 300 x 2,048 x 8,192 34.9 -> 26.3 in three of 64 x 128.
static int slice_k(int K, int slices) { return fw_ceil_div(fw_ceil_div(K, slices), 64) * 64; }

// Bytes of float32 workspace and int32 counters (zero before the first call; left zero) of a product on named tiles; 0 and 0 with one slice. -1: no
// such tile, or it does not take the shape: K a multiple of 32 (up to 2^22; N up to 2^20), with K cut every slice some of it and at least one workgroup a slice.
extern "C" int fw_gemm_mfma_big_tile_needs(int mode, int M, int N, int K, int rows, int columns, int each_cu, int slices, size_t* workspace_bytes, int* counters) {
    FW_REQUIRE(M >= 1 && N > 0 && K > 0 && mode >= 0 && mode <= 2, "gemm_mfma_big_tile: M %d N %d K %d mode %d", M, N, K, mode);
    FW_REQUIRE(slices >= 1 && slices <= B_SLICES && fw_big_tile_exists(mode, rows, columns, each_cu, slices),
               "gemm_mfma_big_tile: no tile of %d x %d in mode %d, %d on a compute unit, K in %d slices", rows, columns, mode, each_cu, slices);
    FW_REQUIRE(K % BK == 0 && K <= BK_MOST && N <= BN_MOST, "gemm_mfma_big_tile: N %d K %d: K a multiple of %d up to %d, N up to %d", N, K, BK, BK_MOST, BN_MOST);
    const long long tiles = (long long)fw_ceil_div(M, rows) * fw_ceil_div(N, mode == MB_SWIGLU ? columns / 2 : columns);
    FW_REQUIRE(tiles * slices < (1ll << 30), "gemm_mfma_big_tile: too many tiles");
    FW_REQUIRE((long long)slice_k(K, slices) * (slices - 1) < K, "gemm_mfma_big_tile: K %d has no %d slices of whole 64 k", K, slices);
    *workspace_bytes = slices > 1 ? (size_t)slices * tiles * rows * columns * sizeof(float) : 0;
    *counters = slices > 1 ? (int)tiles : 0;
    return 0;
}

// fw_gemm_mfma's contract on the tile named. Calls with K cut that overlap on one device must not share counters or workspace.
extern "C" int fw_gemm_mfma_big_tile(const void* a, const void* w, const float* bias, void* out, int out_dtype, int mode, int M, int N, int K, int rows,
                                     int columns, int each_cu, int slices, void* workspace, size_t workspace_bytes, int* counters, int counters_len, void* stream) {
    size_t need_bytes = 0;
    int need_counters = 0;
    if (check_operands(a, w, bias, out_dtype, mode, M, N, K)) return -1;
    if (fw_gemm_mfma_big_tile_needs(mode, M, N, K, rows, columns, each_cu, slices, &need_bytes, &need_counters)) return -1;
    FW_REQUIRE(slices == 1 || (workspace != nullptr && workspace_bytes >= need_bytes && counters != nullptr && counters_len >= need_counters && (uintptr_t)workspace % 16 == 0),
               "gemm_mfma_big_tile: this shape needs %zu bytes of workspace and %d counters", need_bytes, need_counters);
    if (launch(mode, {a, w, bias, out, out_dtype, M, N, K, rows, columns, each_cu, slices, slice_k(K, slices), (float*)workspace, counters, (hipStream_t)stream})) return -1;
    FW_LAUNCH_CHECK("gemm_mfma_big_tile");
    return 0;
}

// The gated product with clamped halves on the tile named: out bfloat16 [M][N] = g sigmoid(alpha g) (u + shift), g = min(gate, limit), u = clamp(up, -limit,
// limit), formed from the float32 sums. The sums in memory and a pass over them took 83 + 23 us of 1,111 x 8,192 over K 2,048, this 75 (tiles of 192 x 128); 277 rows 30 + 6 and 29.
extern "C" int fw_gemm_mfma_big_tile_clamped(const void* a, const void* w, void* out, int M, int N, int K, int rows, int columns, int each_cu, float limit, float alpha,
                                             float shift, void* stream) {
    size_t need_bytes = 0;
    int need_counters = 0;
    if (check_operands(a, w, nullptr, FW_BF16, MB_SWIGLU, M, N, K)) return -1;
    if (fw_gemm_mfma_big_tile_needs(MB_SWIGLU, M, N, K, rows, columns, each_cu, 1, &need_bytes, &need_counters)) return -1;
    FW_REQUIRE(limit > 0.0f, "gemm_mfma_big_tile_clamped: the limit must be positive");
    BigCall call = {a, w, nullptr, out, FW_BF16, M, N, K, rows, columns, each_cu, 1, K, nullptr, nullptr, (hipStream_t)stream};
    call.limit = limit;
    call.alpha = alpha;
    call.shift = shift;
    if (fw_launch_big_clamped(call)) return -1;
    FW_LAUNCH_CHECK("gemm_mfma_big_tile_clamped");
    return 0;
}
