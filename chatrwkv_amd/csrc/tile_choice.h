// The tile and the K split that a launch of the direct-to-LDS contractions (gemm.hip) runs with: host code that needs no GPU.
#pragma once
#include <cstddef>
#include <cstdint>

namespace {

// The direct-to-LDS tiles: rows and columns.  TILE_S is 128 x 128 with three stages (two workgroups fit a CU), TILE_S4 with four
// and K over two groups, TILE_K8 and TILE_K4 gemm_kg_kernel with eight and four groups.
enum {
    TILE_256x256, TILE_S, TILE_S4, TILE_K8, TILE_K4, TILE_256x192, TILE_224x256, TILE_224x192, TILE_192x256, TILE_192x192,
    TILE_160x256, TILE_160x192, TILE_128x256, TILE_128x192,
    TILE_32x16, TILE_32x32, TILE_32x48, TILE_32x64, TILE_32x96, TILE_48x16, TILE_48x32, TILE_48x48, TILE_48x64, TILE_48x96, TILE_64x16, TILE_64x32, TILE_64x48, TILE_64x64, TILE_64x96,
    TILE_96x128, TILE_128x96, TILE_96x96, TILES
};
struct TileDim { int tm, tn; };
constexpr TileDim tile_dim[TILES] = {{256, 256}, {128, 128}, {128, 128}, {64, 64}, {64, 128}, {256, 192}, {224, 256}, {224, 192},
                                     {192, 256}, {192, 192}, {160, 256}, {160, 192}, {128, 256}, {128, 192},
                                     {32, 16}, {32, 32}, {32, 48}, {32, 64}, {32, 96}, {48, 16}, {48, 32}, {48, 48}, {48, 64}, {48, 96}, {64, 16}, {64, 32}, {64, 48}, {64, 64}, {64, 96},
                                     {96, 128}, {128, 96}, {96, 96}};

// Cost model of a direct-to-LDS launch in microseconds.  `tiles` tiles of nk k-tiles split c ways run in rounds over the 256 CUs:
//   launch + rounds * (round, or split_round, which leaves the epilogue to the second pass)
//          + k-tiles * (step_1 for every full round, between step_0 and step_1 for the last one by the CUs busy,
//                       extra for what exceeds one round)
//          + with a split, slab per 16 MB of fp32 slabs written and read, split per slab, and SECOND_LAUNCH.
// No term is below 0, and they make up for each other: one by itself, several being 0, is no cost of the hardware.
// One fit per tile and type, over launches within 1.6 times the best one of 648 products each (24 lengths from 17 to 2048 rows, 27 widths
// from 64 to 20480; weights from HBM; the chip under load before): the tile and split it picks takes 1 % (uint8) and 2 %
// (fp16) longer than the best of all on average, with products that the host launches no faster counted in.  A tile per round costs
// between 3 and 15 us whatever K is, so tiles of many sizes pay: each of these is the choice somewhere (64 x 16 with fp16 weights alone), the large ones with sides of
// 160, 192 and 224 where 256 x 256 or 128 x 128 leave CUs idle or rows empty, those of 32, 48 and 64 rows in calls of up to 128 rows, those with a side of
// 96 where a round of 128 x 128 leaves CUs idle (fitted apart, at full depth, 97 rows and more).
// us, uint8 / fp16 weights: [1024 x 4096] x [4096 x 12288] three rounds of 128 x 128 115.7 / 132.5, one of 256 x 192 90 / 97; [777 x
// 4096] x [4096 x 16384] 256 x 256 126 / 130, 224 x 256 100 / 107; [768 x 4096] x [4096 x 12288] 104 / 109, 192 x 192 71 / 80;
// [45 x 4096] x [4096 x 4096] four splits of 64 x 64 11.0 / 12.4, 48 x 16 at full depth 8.7 / 10.6; [45 x 4096] x [4096 x 20480] 64 x 128 26.5 /
// 40.6, 48 x 96 23.8 / 37.9; [24 x 2048] x [2048 x 2048] 8.1 / 8.1, 32 x 16 5.6 / 5.5; [333 x 2048]
// x [2048 x 8192] four-stage 128 x 128 21.5 / 22.8, 96 x 128 19.1 / 20.2; [160 x 4096] x [4096 x 16384] 40.5 / 44.0, 33.5 / 42.7; [513 x
// 4096] x [4096 x 4096] 33.0 / 31.8, 128 x 96 28.9 / 29.7; [513 x 1280] x [1280 x 3840] 16.1 / 14.3, 96 x 96 12.4 / 12.0.
// A split's second launch was measured again as part of a chain of launches (graphs of 4 to 24 of them, each on weights of its own; 952 products of
// 17 to 513 rows per type, up to 16 candidates each): the splits of 32 x 16 took 0.9 / 0.55 us more than fitted beside the other
// tiles, all splits together 0.2.  With both in the prices the choice for those products takes 0.9 / 2.4 % longer than the best candidate,
// 1.1 / 2.7 before (and 1.0 / 2.5 or 1.5 / 2.8 with 0.5 or 2 us on every split instead).  us, scaling pass included: uint8 [24 x 3072] x [3072
// x 768] two splits 9.8, full depth 9.0; [17 x 4096] x [4096 x 2048] 10.6, 9.7; [45 x 4096] x [4096 x 4096] 48 x 32 in two splits 14.6, 48 x 16 14.2;
// fp16 [17 x 3072] x [3072 x 768] 7.1, 6.3.  [513 x 3072] x [3072 x 768], 64 x 64, two splits / full depth: uint8 17.8 both, fp16 12.3 / 12.6.
constexpr float SECOND_LAUNCH = 0.2f;
struct TilePrice { float launch, round, split_round, step_0, step_1, extra, slab, split; };
constexpr TilePrice tile_price[2][TILES] = {
    {   // fp16 weights
        {4.549f, 9.813f, 10.035f, 0.941f, 1.721f, 0.081f, 3.477f, 0.f},   // 256x256
        {2.456f, 3.248f, 4.838f, 0.423f, 0.631f, 0.f, 4.568f, 0.076f},   // S
        {1.871f, 4.556f, 4.704f, 0.298f, 0.575f, 0.f, 7.450f, 0.136f},   // S4
        {1.987f, 2.281f, 4.023f, 0.141f, 0.253f, 0.f, 4.754f, 0.175f},   // K8
        {1.808f, 3.209f, 4.405f, 0.217f, 0.391f, 0.f, 7.476f, 0.162f},   // K4
        {4.715f, 8.832f, 6.523f, 0.825f, 1.348f, 0.067f, 4.078f, 0.019f},   // 256x192
        {5.750f, 7.778f, 9.926f, 0.869f, 1.545f, 0.f, 2.620f, 0.f},   // 224x256
        {5.169f, 7.209f, 5.179f, 0.704f, 1.218f, 0.005f, 4.432f, 0.f},   // 224x192
        {5.462f, 5.451f, 8.367f, 0.833f, 1.404f, 0.034f, 2.485f, 0.067f},   // 192x256
        {6.233f, 4.192f, 4.042f, 0.576f, 1.135f, 0.013f, 3.789f, 0.014f},   // 192x192
        {5.662f, 4.463f, 7.448f, 0.729f, 1.266f, 0.f, 2.506f, 0.064f},   // 160x256
        {6.807f, 2.897f, 4.219f, 0.444f, 1.116f, 0.f, 2.900f, 0.f},   // 160x192
        {3.811f, 5.068f, 6.800f, 0.674f, 1.048f, 0.f, 4.031f, 0.006f},   // 128x256
        {3.662f, 4.895f, 5.956f, 0.520f, 0.831f, 0.015f, 3.948f, 0.f},   // 128x192
        {2.064f, 1.754f, 2.120f, 0.045f, 0.071f, 0.029f, 8.577f, 0.499f},   // 32x16
        {3.459f, 0.f, 0.708f, 0.075f, 0.127f, 0.004f, 0.f, 0.356f},   // 32x32
        {2.995f, 1.030f, 2.668f, 0.077f, 0.169f, 0.031f, 0.f, 0.107f},   // 32x48
        {2.020f, 1.586f, 3.023f, 0.107f, 0.209f, 0.002f, 0.f, 0.249f},   // 32x64
        {2.242f, 1.739f, 3.490f, 0.122f, 0.309f, 0.f, 1.050f, 0.125f},   // 32x96
        {2.035f, 1.839f, 2.184f, 0.066f, 0.101f, 0.019f, 5.215f, 0.412f},   // 48x16
        {3.611f, 0.f, 0.981f, 0.097f, 0.180f, 0.f, 0.f, 0.295f},   // 48x32
        {3.170f, 1.064f, 2.539f, 0.091f, 0.237f, 0.019f, 6.597f, 0.109f},   // 48x48
        {2.941f, 0.957f, 2.587f, 0.118f, 0.329f, 0.f, 2.137f, 0.100f},   // 48x64
        {3.241f, 1.435f, 2.964f, 0.140f, 0.488f, 0.f, 2.435f, 0.047f},   // 48x96
        {3.061f, 0.871f, 1.378f, 0.080f, 0.124f, 0.043f, 0.f, 0.407f},   // 64x16
        {3.389f, 0.364f, 1.904f, 0.101f, 0.197f, 0.061f, 0.317f, 0.153f},   // 64x32
        {4.503f, 0.040f, 1.948f, 0.095f, 0.337f, 0.117f, 0.f, 0.027f},   // 64x48
        {2.451f, 1.661f, 3.319f, 0.136f, 0.330f, 0.f, 4.174f, 0.119f},   // 64x64
        {2.816f, 2.220f, 3.033f, 0.188f, 0.429f, 0.f, 7.091f, 0.094f},   // 64x96
        {1.795f, 4.124f, 4.124f, 0.260f, 0.484f, 0.002f, 0.f, 0.f},   // 96x128
        {1.738f, 4.854f, 4.854f, 0.263f, 0.457f, 0.039f, 0.f, 0.f},   // 128x96
        {1.881f, 4.025f, 4.025f, 0.246f, 0.404f, 0.029f, 0.f, 0.f},   // 96x96
    }, {   // uint8
        {5.336f, 9.067f, 8.377f, 0.949f, 1.642f, 0.022f, 3.336f, 0.f},   // 256x256
        {6.522f, 0.f, 0.599f, 0.349f, 0.546f, 0.f, 4.631f, 0.085f},   // S
        {3.456f, 3.989f, 3.830f, 0.317f, 0.523f, 0.041f, 5.040f, 0.081f},   // S4
        {1.922f, 3.185f, 4.514f, 0.115f, 0.176f, 0.013f, 6.113f, 0.121f},   // K8
        {1.799f, 3.765f, 4.212f, 0.200f, 0.305f, 0.021f, 7.262f, 0.149f},   // K4
        {5.813f, 9.209f, 4.665f, 0.786f, 1.222f, 0.067f, 4.361f, 0.f},   // 256x192
        {6.485f, 8.992f, 8.275f, 0.837f, 1.443f, 0.027f, 2.592f, 0.f},   // 224x256
        {5.976f, 8.521f, 5.926f, 0.677f, 1.123f, 0.072f, 3.349f, 0.f},   // 224x192
        {5.631f, 7.400f, 8.116f, 0.702f, 1.282f, 0.041f, 2.417f, 0.089f},   // 192x256
        {5.123f, 7.379f, 3.369f, 0.573f, 0.988f, 0.088f, 4.369f, 0.092f},   // 192x192
        {5.432f, 6.626f, 6.901f, 0.678f, 1.133f, 0.029f, 2.803f, 0.050f},   // 160x256
        {6.671f, 4.130f, 4.142f, 0.495f, 0.891f, 0.104f, 3.467f, 0.f},   // 160x192
        {6.383f, 3.449f, 3.229f, 0.589f, 0.939f, 0.128f, 3.964f, 0.092f},   // 128x256
        {6.019f, 3.214f, 3.148f, 0.518f, 0.752f, 0.093f, 4.309f, 0.040f},   // 128x192
        {1.699f, 2.323f, 2.958f, 0.041f, 0.055f, 0.f, 12.951f, 0.432f},   // 32x16
        {3.999f, 0.f, 0.899f, 0.066f, 0.083f, 0.004f, 2.289f, 0.215f},   // 32x32
        {2.913f, 1.532f, 3.101f, 0.071f, 0.098f, 0.023f, 2.608f, 0.078f},   // 32x48
        {4.114f, 0.f, 1.196f, 0.086f, 0.112f, 0.015f, 3.985f, 0.176f},   // 32x64
        {3.385f, 1.010f, 2.444f, 0.122f, 0.163f, 0.054f, 6.361f, 0.100f},   // 32x96
        {4.058f, 0.069f, 1.352f, 0.059f, 0.074f, 0.028f, 8.241f, 0.155f},   // 48x16
        {4.037f, 0.f, 0.851f, 0.079f, 0.097f, 0.028f, 2.529f, 0.277f},   // 48x32
        {4.127f, 0.628f, 2.240f, 0.092f, 0.127f, 0.097f, 5.425f, 0.035f},   // 48x48
        {4.308f, 0.f, 1.565f, 0.115f, 0.151f, 0.106f, 7.660f, 0.069f},   // 48x64
        {4.278f, 0.820f, 2.197f, 0.129f, 0.229f, 0.081f, 5.005f, 0.020f},   // 48x96
        {4.043f, 0.282f, 1.457f, 0.076f, 0.091f, 0.003f, 12.132f, 0.137f},   // 64x16
        {4.251f, 0.f, 1.418f, 0.100f, 0.124f, 0.088f, 6.335f, 0.096f},   // 64x32
        {4.608f, 0.525f, 1.966f, 0.106f, 0.147f, 0.088f, 4.921f, 0.074f},   // 64x48
        {4.535f, 0.f, 1.492f, 0.129f, 0.173f, 0.093f, 8.795f, 0.060f},   // 64x64
        {5.097f, 0.529f, 1.525f, 0.160f, 0.257f, 0.103f, 6.215f, 0.071f},   // 64x96
        {1.500f, 4.811f, 4.811f, 0.295f, 0.412f, 0.026f, 0.f, 0.f},   // 96x128
        {1.500f, 5.567f, 5.567f, 0.284f, 0.397f, 0.026f, 0.f, 0.f},   // 128x96
        {4.415f, 1.814f, 1.814f, 0.238f, 0.325f, 0.016f, 0.f, 0.f},   // 96x96
    }};
// The same by field, for loops over the tiles.
struct Prices { float launch[TILES], round[TILES], split_round[TILES], step_0[TILES], step_1[TILES], extra[TILES], slab[TILES], split[TILES]; };
constexpr Prices by_field(const TilePrice (&p)[TILES]) {
    Prices f{};
    for (int t = 0; t < TILES; ++t) {
        f.launch[t] = p[t].launch; f.round[t] = p[t].round; f.split_round[t] = p[t].split_round; f.step_0[t] = p[t].step_0;
        f.step_1[t] = p[t].step_1; f.extra[t] = p[t].extra; f.slab[t] = p[t].slab; f.split[t] = p[t].split;
    }
    return f;
}
constexpr Prices prices[2] = {by_field(tile_price[0]), by_field(tile_price[1])};

// The launches that a tile is offered for: those it was measured in.  The tiles with a side of 96 in calls of 65 to 96 rows, one row of tiles,
// where they nearly fill a round: us, scaling pass included, at 80 or 96 rows with them / with the best choice among the others / with the one
// that was taken, uint8 [4096] x [4096 x 20480], 214 of them, 37.4 / 39.6 / 44.0, [2048] x [2048 x 18432], 192, 22.3 / 24.2 / 25.8, fp16 47.2 / 50.1 / 51.0 and
// 24.7 / 26.1 / 27.0; the 32768 outputs of 256 of 96 x 128 48.0 / 49.5.  With fewer the others are faster by more than the
// prices say, uint8 [4096] x [4096 x 14336], 150, 34.7 / 28.7, [4096 x 12288] 34.4 / 26.0, [4096 x 4096] 32.8 / 16.2, and so they are past a
// round, [2048] x [2048 x 50304] 44.7 / 42.1.  5120 inputs, fp16, 65 rows: up to 3 % slower with them, at 96 rows 8 % faster.
inline bool tile_offered(int tile, int64_t T, float tiles) {
    if (tile >= TILE_96x128) return T > 96 || (T > 64 && tiles >= 192.f && tiles <= 256.f);
    if (tile >= TILE_32x16) return T <= (tile_dim[tile].tn <= 32 ? 128 : 256);
    return true;
}

struct TilePick { int tile, ks; float us; };
constexpr float NEVER = 1e30f;

// A launch to choose for: n products of T rows, nk k-tiles and M_i outputs, with ws_bytes for slabs.  A choice is made per launch, up to
// ten times a layer, and the host is the slower side of small models and of short products.  So there are no divisions but by
// constants, and the prices of all tiles come from loops without branches: 0.33 us a choice where tile after tile and split after split
// took 0.9 (uint8 [45 x 768] x [768 x 3072] by the operator, one call after the other, 17.5 -> 16.6 us).
class Launch {
    static constexpr int SIDES = 17;                 // by the side in units of 16
    int64_t T;
    int rows[SIDES], cols[SIDES];
    int splits;
    float ways[8], depth[8], out16;                  // K splits: 1 to 8, whole k-tiles, at least 8 per split, slabs within ws_bytes; slabs in 16 MB

  public:
    Launch(int64_t T, int nk, int n, const int64_t *M, size_t ws_bytes) : T(T), splits(0) {
        count<true>(T, rows);
        count<true>(M[0], cols);
        for (int i = 1; i < n; ++i) count<false>(M[i], cols);
        uint64_t out_bytes = 0;
        for (int i = 0; i < n; ++i) out_bytes += (uint64_t)(T * M[i]) * sizeof(float);
        out16 = (float)out_bytes / (float)(16 << 20);
        for (int c = 1; c <= 8; ++c) {
            if (c > 1 && (nk % c || nk / c < 8 || c * out_bytes > ws_bytes)) continue;
            ways[splits] = (float)c;
            depth[splits++] = (float)(nk / c);
        }
    }
    // `tile` with the K split of least cost, at full depth where it is not offered
    TilePick with(bool w_u8, int tile) const {
        if (!tile_offered(tile, T, tiles(tile))) return {tile, 1, NEVER};
        float us[TILES], ks[TILES];
        price(prices[w_u8], tile, tile + 1, us, ks);
        return {tile, (int)ks[tile], us[tile]};
    }
    // the tile of least cost among those offered
    TilePick best(bool w_u8) const {
        float us[TILES], ks[TILES];
        const Prices &p = prices[w_u8];
        const int few = T <= 256 ? TILE_96x128 : TILE_32x16;
        price(p, 0, few, us, ks);
        price(p, TILE_96x128, TILES, us, ks);
        TilePick b = {TILE_S, 1, NEVER};
        for (int t = 0; t < TILES; t = t + 1 == few ? TILE_96x128 : t + 1)
            if (us[t] < b.us && tile_offered(t, T, tiles(t))) b = {t, (int)ks[t], us[t]};
        return b;
    }

  private:
    float tiles(int t) const { return (float)rows[tile_dim[t].tm >> 4] * (float)cols[tile_dim[t].tn >> 4]; }
    // prices of the tiles [from, to) with their best K splits.  The tiles with a side of 96 run at full depth only: split they were the
    // best of all, by 5 % at most, for 6 of 560 products, and priced for it they took others where they are 10 to 15 % slower.
    void price(const Prices &p, int from, int to, float *us, float *ks) const {
        float n[TILES];
        for (int t = from; t < to; ++t) {
            n[t] = tiles(t);
            us[t] = NEVER;
            ks[t] = 1.f;
        }
        for (int s = 0; s < (from >= TILE_96x128 ? 1 : splits); ++s) {
            const float c = ways[s], d = depth[s];
            const float *round = s ? p.split_round : p.round;
            for (int t = from; t < to; ++t) {
                const float wgs = n[t] * c, x = wgs * (1.f / 256.f), rounds = (float)(int)((wgs + 255.f) * (1.f / 256.f));
                float k = p.launch[t] + rounds * round[t] + d * p.step_1[t] * x + d * p.step_0[t] * (rounds - x) + d * p.extra[t] * (x > 1.f ? x - 1.f : 0.f);
                k += s ? SECOND_LAUNCH + c * (p.split[t] + p.slab[t] * out16) : 0.f;
                ks[t] = k < us[t] ? c : ks[t];
                us[t] = k < us[t] ? k : us[t];
            }
        }
    }
    template <bool FIRST, int SIDE>
    static void count_side(uint32_t n, int *out) {
        const int k = (int)((n + (SIDE - 1)) / SIDE);
        out[SIDE / 16] = FIRST ? k : out[SIDE / 16] + k;
    }
    template <bool FIRST>
    static void count(int64_t n, int *out) {         // tiles along n <= 2^24
        const uint32_t m = (uint32_t)n;
        count_side<FIRST, 16>(m, out); count_side<FIRST, 32>(m, out); count_side<FIRST, 48>(m, out); count_side<FIRST, 64>(m, out);
        count_side<FIRST, 96>(m, out); count_side<FIRST, 128>(m, out); count_side<FIRST, 160>(m, out); count_side<FIRST, 192>(m, out);
        count_side<FIRST, 224>(m, out); count_side<FIRST, 256>(m, out);
    }
};

}  // namespace
