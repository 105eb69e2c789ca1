// The grouped GEMM with tiles of 256 x 256, one workgroup of 8 waves per compute unit, and what all tile sizes share.
#define MOE_GEMM_TILE 256
#include "grouped_gemm_kernel.h"


// The gate/up pair kernel never splits K: it holds two products and is at its limit of registers without an exchange (a launch of 3.5 rounds, as 8
// experts of f = 14336 and at most 256 rows make, leaves half of the chip idle in its last).  The others may cut the tiles of the last, partial round of
// compute units 2 or 4 ways.
int moe_gemm_max_split(bool pair) { return pair ? 1 : 4; }
int moe_gemm_cus()
{
    const int n = moe_device_cus() / NXCD * NXCD;
    return n < NXCD ? NXCD : n;
}

int64_t moe_gemm_plan_blocks(int tile, int64_t R, int E, int64_t N, int pair) { return tile == 128 ? moe_gemm_small_plan_blocks(R, E, N, pair) : plan_blocks(R, E, N, pair); }
int moe_launch_gemm_plan(int tile, const void* offsets, int off64, int E, int64_t R, int64_t K, int64_t N, int pair, int nseg, int* out, hipStream_t stream)
{
    if (K < BK || nseg < 1 || nseg > 2) return MOE_ERR_UNSUPPORTED;
    return tile == 128 ? moe_launch_gemm_small_plan(offsets, off64, E, R, K, N, pair, nseg, out, stream) : launch_plan(offsets, off64, E, R, K, N, pair, nseg, out, stream);
}

// exchange area of a launch: one counter per split tile and one fp32 partial tile per split item; at most one round
// of compute units' worth of either
size_t moe_gemm_sk_bytes(int cus, int64_t R, int E, int64_t N)
{
    size_t bytes = 0;   // of the tile size that needs more
    for (int tile = 256; tile >= 128; tile /= 2) {
        const int64_t tiles = (R / tile + E) * ((N + tile - 1) / tile), most = 256 / tile * cus;
        const size_t b = (size_t)(4 * tiles < most ? 4 * tiles : most) * tile * tile * sizeof(float);
        bytes = b > bytes ? b : bytes;
    }
    return (size_t)cus * sizeof(int) + 256 + bytes;
}

// what a launch of these sizes (K: all segments) and tiles writes of that area behind the counters, at most
size_t moe_gemm_exchange_bytes(int cus, int tile, int64_t R, int E, int64_t K, int64_t N)
{
    const int64_t tiles = (R / tile + E) * ((N + tile - 1) / tile), most = 256 / tile * cus;
    int64_t split = 1;
    while (split * 2 <= moe_gemm_max_split(false) && (K + BK - 1) / BK / (split * 2) >= MIN_PART_KTILES) split *= 2;
    return split == 1 ? 0 : (size_t)(split * tiles < most ? split * tiles : most) * tile * tile * sizeof(float);
}

void moe_gemm_sk_attach(MoeGemmParams& p, void* ws, int cus)
{
    p.num_cus = cus;
    p.sk_counters = (int*)ws;
    p.sk_partials = (float*)((uint8_t*)ws + (((size_t)cus * sizeof(int) + 255) & ~(size_t)255));
}

bool moe_gemm_mfma_supported(const MoeGemmParams& p, int64_t R)
{
    auto al16 = [](const void* q) { return q == nullptr || ((uintptr_t)q % 16) == 0; };
    // whole 64-wide K tiles run through the main loop (at least one), a remainder (multiple of 8) through the tail step
    if (p.K < BK || p.K % 8 != 0 || p.N % 8 != 0 || p.ldx % 8 != 0 || p.ldw % 8 != 0 || p.swe % 8 != 0) return false;
    if (!al16(p.X[0]) || !al16(p.X[1]) || !al16(p.W[0]) || !al16(p.W[1])) return false;
    for (int i = 0; i < MOE_MAX_SLABS; ++i)
        if (!al16(p.Q[i]) || !al16(p.LB[i])) return false;   // (slabs beyond these: multiples of 16 bytes from Q[0] / LB[0], checked below)
    if (p.nseg < 1 || p.nseg > 2 || (p.nseg == 2 && p.epi != MOE_EPI_STORE) || p.nslab < 0 || (p.slab_mode == 1 && p.nslab % 2 != 0)) return false;
    if (p.K % BK != 0 && p.epi != MOE_EPI_STORE) return false;   // a partial last K tile: the plain epilogue only
    if (p.nslab > MOE_MAX_SLABS) {
        const bool epi_ok = p.epi == MOE_EPI_STORE || (!p.nn && (p.epi == MOE_EPI_SWIGLU || p.epi == MOE_EPI_SWIGLU_BWD));
        if (!epi_ok || (p.slab_mode == 1) != (p.epi == MOE_EPI_SWIGLU) || p.nslab > MOE_MAX_STRIDED_SLABS || p.q_slab_stride % 8 != 0 || p.lb_slab_stride % 8 != 0) return false;
    }
    // 32-bit byte offsets: gathered A rows from the start of X (grouped ones from the tile's first row), weights from
    // the start of one expert's matrix, grouped outputs and the saved gate / up from the tile's first row; scattered
    // output rows from the start of Y while Y spans less than 2 GiB, 64-bit addresses beyond (y_wide, set at launch)
    (void)R;
    const int fo = p.fan_out > 0 ? p.fan_out : 1;
    const int64_t x_rows = p.x_grouped ? BM : (R + fo - 1) / fo;
    // (a partial last K tile masks its loads through the descriptor's range, which that kernel variant sets to 2 GiB)
    const int64_t limit = (p.K % BK != 0) ? (int64_t)1 << 31 : (int64_t)1 << 32;
    if ((x_rows * p.ldx + p.K) * 2 >= limit) return false;
    if (((p.nn ? p.K : p.N) * p.ldw + (p.nn ? p.N : p.K)) * 2 >= limit) return false;
    if ((BM * p.ldy + p.N) * 2 >= ((int64_t)1 << 31)) return false;
    if ((p.epi == MOE_EPI_SWIGLU_BWD || p.epi == MOE_EPI_SWIGLU_BWD_FUSED) && (BM * p.ldh + p.N) * 2 >= ((int64_t)1 << 31)) return false;
    return true;
}

// A launch whose 256 x 256 tiles, split along K as far as they may be, take at most half of the compute units is latency: look-up, first loads, a chain of K tiles and
// an epilogue on workgroups of which most of the chip has none.  Quarter tiles spread it over up to four times as many workgroups, each with a quarter of the
// epilogue.  Launches in us with large and small tiles: 512 tokens, d = 256, f = 512, 8 experts: gate/up (36 workgroups) 15.8 and 12.9, h W2 16.0 and 12.4, dh 24.2 and 16.3, dX 21.4
// and 16.0; 64 rows of one expert, d = 4096, f = 14336: gate/up (112) 59.8 and 46.3, h W2 (64) 55.9 and 44.9, dh (224) 46.7 and 54.0, dX (64) 97 and 82; 500 rows: gate/up (224) 98
// and 142, h W2 (128) 93 and 98, dX (128) 159 and 154 (319 rows, all of it 409 and 419); 2 rows of two experts: h W2 (128) 52 and 49; 4 tokens: h W2 (224) 115 and 142.  Groups of more than 128 rows
// fetch their weights for more row tiles, so they take small tiles up to three eighths of the chip only.  Where the chip is full the small tiles fetch
// twice the operand bytes per product: 2048 tokens, 64 experts, top-8 837 us and 946.
//
// The second condition is for rows that are not dealt evenly, which the host does not see: a group of 129 rows is two small tiles and one large one.  Two small tiles on one
// compute unit take as long as a large one there, so of a launch that splits K the small ones must come to at most one per compute unit however the rows fall.  Of
// 5000 drawn products (128 to 14336 columns and deep, 1 to 96 groups), small tiles by the first condition alone: those whose tiles came to one at most 0.95-1.93 times as fast as large ones,
// those of more 0.77-1.37, 28 % of them slower by more than 1.5 %: us, large and small, 64 groups of 121 rows on average, 1408 x 192 31.1 and 40.3; 16 of 140, 1216 x 768 30.1 and 36.6; 32 of
// 123, 3968 x 256 57.2 and 66.7; dX of two groups of 126, 28672 x 4096, and the kernels around it 210 and 245.  Launches that never split have a longer chain of K tiles to lose on the idle half: up to
// one and a half per compute unit (gate/up of 16 groups, 124 rows on average, 2816 x 960 and the kernels behind it 93.6 and 97.1 with 1.8; 1.05-1.6 times as fast up to 1.5).
int moe_gemm_tile(int cus, int64_t R, int E, int64_t K, int64_t N, bool pair)
{
    if (R < 1 || K % BK != 0) return 256;
    const int64_t groups = R < E ? R : E, ncu = cus;
    const int64_t tiles = groups * (((R + groups - 1) / groups + BM - 1) / BM) * ((N + BN - 1) / BN * (pair ? 2 : 1));   // (as if the rows were dealt evenly)
    int64_t split = 1, parts = 1;
    while (split * 2 <= moe_gemm_max_split(pair) && tiles * split * 2 <= ncu && K / BK / (split * 2) >= MIN_PART_KTILES) split *= 2;
    if (R <= groups * 128 ? tiles * split * 2 > ncu : tiles * split * 8 > 3 * ncu) return 256;
    while (parts * 2 <= moe_gemm_max_split(pair) && K / BK / (parts * 2) >= MIN_PART_KTILES) parts *= 2;
    const int64_t small = (groups + (R - groups) / 128) * (pair ? (N + 63) / 64 : (N + 127) / 128) * parts;   // at most, however the rows fall
    return 2 * small <= (parts > 1 ? 2 : 3) * ncu ? 128 : 256;
}

static std::atomic<int64_t> g_mfma_launches{0};
int64_t moe_gemm_mfma_launch_count() { return g_mfma_launches; }

int moe_launch_gemm_mfma(const MoeGemmParams& p, int64_t R, hipStream_t stream)
{
    if (R == 0 || p.N == 0) return MOE_OK;
    if (!moe_gemm_mfma_supported(p, R)) return MOE_ERR_UNSUPPORTED;
    ++g_mfma_launches;
    const bool general = p.K % BK != 0 || p.nslab > MOE_MAX_SLABS;   // (the variants for these have one tile size)
    if (p.tile != 0 && p.tile != 128 && p.tile != 256) return MOE_ERR_BAD_ARG;
    if (general && p.tile == 128) return MOE_ERR_UNSUPPORTED;
    const int tile = p.tile ? p.tile : general ? 256 : moe_gemm_tile(p.num_cus ? p.num_cus : moe_gemm_cus(), R, p.E, p.K * p.nseg, p.N, EPI_IS_PAIR(p.epi));
    if (tile == 128) return moe_launch_gemm_small_tile(p, R, stream);
    return launch_epilogue(p, R, stream);
}
