// 3x3 stride-1 tile variants of the MFMA conv kernel (conv_kernel.hpp).

#include "conv_ws.hpp"

namespace mlvc_hip {
namespace conv {

namespace {
const Variant kTable[] = {
    MLVC_VARIANT_OCC(32, 4, 64, 3, 3, 1, 16, 4),
    costed(with_ragged<32, 8, 32, 3, 3, 1, 16, 1, 4, 4>(MLVC_VARIANT_OCC(32, 8, 32, 3, 3, 1, 16, 4)), 1.578f, 0.607f, 1.408f, 0.439f),
    MLVC_VARIANT_OCC(64, 4, 32, 3, 3, 1, 16, 4),
    MLVC_VARIANT_S2D(32, 4, 64, 3, 3, 1, 16),
    MLVC_VARIANT_S2D(32, 8, 32, 3, 3, 1, 16),
    MLVC_VARIANT_S2D(64, 4, 64, 3, 3, 1, 16),
    MLVC_VARIANT_S2D(64, 8, 32, 3, 3, 1, 16),
    MLVC_VARIANT(64, 16, 16, 3, 3, 1, 16),
    MLVC_VARIANT(64, 2, 64, 3, 3, 1, 16),
    MLVC_VARIANT_S2D(64, 4, 32, 3, 3, 1, 16),
    MLVC_VARIANT_S2D(64, 8, 16, 3, 3, 1, 16),
    MLVC_VARIANT(128, 4, 64, 3, 3, 1, 16),
    MLVC_VARIANT(128, 8, 32, 3, 3, 1, 16),
    MLVC_VARIANT_W(128, 16, 32, 3, 3, 1, 16, 1, 8),
    MLVC_VARIANT_W(128, 8, 64, 3, 3, 1, 16, 1, 8),
    MLVC_VARIANT_W(256, 8, 32, 3, 3, 1, 16, 2, 4),
    MLVC_VARIANT_W(256, 4, 64, 3, 3, 1, 16, 2, 4),
    MLVC_VARIANT_W(64, 16, 32, 3, 3, 1, 16, 1, 8),
    MLVC_VARIANT_W(128, 16, 16, 3, 3, 1, 16, 2, 4),
    MLVC_VARIANT(128, 16, 16, 3, 3, 1, 16),
    MLVC_VARIANT(32, 8, 32, 3, 3, 1, 32),
    MLVC_VARIANT(64, 8, 32, 3, 3, 1, 32),
    MLVC_VARIANT(64, 4, 64, 3, 3, 1, 32),
    MLVC_VARIANT(64, 8, 16, 3, 3, 1, 32),
    MLVC_VARIANT_DB(64, 8, 32, 3, 3, 1, 16),
    MLVC_VARIANT_DB(32, 8, 32, 3, 3, 1, 16),
    MLVC_VARIANT_DB(128, 8, 32, 3, 3, 1, 16),
    MLVC_VARIANT_DB(128, 4, 64, 3, 3, 1, 16),
    MLVC_VARIANT_DB(64, 4, 64, 3, 3, 1, 16),
    costed(MLVC_VARIANT_OCC(32, 2, 64, 3, 3, 1, 16, 4), 2.179f, 0.678f, 0.959f, 0.314f),
    costed(MLVC_VARIANT_WO(32, 2, 32, 3, 3, 1, 16, 1, 2, 4), 2.555f, 0.680f, 0.416f, 0.255f),
    MLVC_VARIANT_WO(64, 2, 32, 3, 3, 1, 16, 1, 2, 4),
    MLVC_VARIANT_WS(256, 4, 32, 128, 2),
    MLVC_VARIANT_WS(128, 4, 32, 128, 2),
    MLVC_VARIANT_WS(256, 4, 32, 64, 2),
    costed(with_ragged_ws<WsCfg<128, 4, 32, 64, 2>>(MLVC_VARIANT_WS(128, 4, 32, 64, 2)), 1.602f, 0.469f, 2.396f, 0.948f),
    costed(with_ragged_ws<WsCfg<256, 2, 32, 128, 2>>(MLVC_VARIANT_WS(256, 2, 32, 128, 2)), 3.523f, 0.068f, 0.942f, 1.137f),
    MLVC_VARIANT_WSR(128, 4, 32, 64, 2, 9),
    MLVC_VARIANT_WSR(256, 2, 32, 128, 2, 9),
    // Widths that divide 120 and 240 (24, 40) or 240 and 480 (48), so the
    // 68x120 and 136x240 decoder convs run without padded columns.
    costed(with_ragged_ws<WsCfg<128, 4, 24, 64, 2, 1, 4, 9>>(MLVC_VARIANT_WSR(128, 4, 24, 64, 2, 9)), 0.773f, 0.665f, 2.488f, 0.605f),
    MLVC_VARIANT_WSR(128, 8, 24, 64, 2, 9),
    costed(with_scalar_ws<WsCfg<128, 4, 40, 64, 2, 1, 4, 9>>(MLVC_VARIANT_WSR(128, 4, 40, 64, 2, 9)), 1.685f, 0.113f, 4.052f, 1.204f),
    MLVC_VARIANT_WSR(128, 4, 48, 64, 2, 9),
    costed(with_scalar_ws<WsCfg<128, 8, 32, 64, 2>>(MLVC_VARIANT_WS(128, 8, 32, 64, 2)), 2.118f, 0.216f, 4.243f, 1.777f),
    // Two m-tiles per wave with a 9-step ring.
    MLVC_VARIANT_WSR(256, 4, 24, 64, 2, 9),
    MLVC_VARIANT_WSR(256, 2, 48, 64, 2, 9),
    // Pipelined passes of 32 channels.
    costed(with_scalar_ws<WsCfg<256, 4, 32, 32, 2>>(MLVC_VARIANT_WSP(256, 4, 32, 32, 2, 3)), 2.936f, 0.292f, 0.731f, 2.101f),
    MLVC_VARIANT_WSP(128, 8, 32, 32, 2, 3),
    MLVC_VARIANT_WSP(128, 4, 32, 32, 2, 9),
    MLVC_VARIANT_WSP(128, 4, 48, 32, 2, 9),
    MLVC_VARIANT_WSP(128, 4, 24, 32, 2, 9),
    // 64 output channels on two waves, more workgroups per CU.
    costed(with_ragged_ws<WsCfg<64, 2, 32, 64, 4, 1, 2, 9>>(MLVC_VARIANT_WSW(64, 2, 32, 64, 4, 2, 9)), 1.364f, 0.838f, 1.451f, 0.179f),
    MLVC_VARIANT_WSW(64, 4, 32, 64, 3, 2, 9),
    MLVC_VARIANT_WSW(64, 8, 32, 64, 2, 2, 9),
    // Short, narrow tiles: enough workgroups for deep convs over few pixels
    // (46x80 and 92x160 planes).
    costed(with_ragged_ws<WsCfg<64, 2, 16, 64, 4, 1, 2, 9>>(MLVC_VARIANT_WSW(64, 2, 16, 64, 4, 2, 9)), 1.102f, 0.727f, 0.873f, 0.122f),
    MLVC_VARIANT_WSR(128, 2, 16, 64, 2, 9),
    // A ring two 16-channel steps deep (18 fragments), for grids of few
    // workgroups: each one's weight stream is then a chain of L2 latencies, a
    // ring of 9 long. One wave of 32 channels for outputs of that few.
    costed(with_ragged_ws<WsCfg<64, 2, 16, 64, 2, 1, 2, 18>>(MLVC_VARIANT_WSW(64, 2, 16, 64, 2, 2, 18)), 1.207f, 0.648f, 1.095f, 0.109f),
    costed(with_ragged_ws<WsCfg<128, 2, 16, 64, 2, 1, 4, 18>>(MLVC_VARIANT_WSR(128, 2, 16, 64, 2, 18)), 0.512f, 0.546f, 1.662f, 0.283f),
    costed(with_ragged_ws<WsCfg<128, 4, 16, 64, 2, 1, 4, 18>>(MLVC_VARIANT_WSR(128, 4, 16, 64, 2, 18)), 0.529f, 0.513f, 2.118f, 0.517f),
    costed(with_ragged_ws<WsCfg<32, 2, 32, 64, 2, 1, 1, 18>>(MLVC_VARIANT_WSW(32, 2, 32, 64, 2, 1, 18)), 2.556f, 0.739f, 1.030f, 0.113f),
    // 512 output channels at 136x240 in one round of two workgroups per CU:
    // 255 8x16 tiles x 2 channel blocks = 510 workgroups, where the 4x48
    // tiles' 680 take two rounds of 512 slots with the second a third full.
    // LDS for the channel-last DEPTH_TO_SPACE(2) output tile (72 KB).
    costed(with_scalar_ws<WsCfg<256, 8, 16, 32, 2>>(MLVC_VARIANT_WSPD(256, 8, 16, 32, 2, 3)), 2.934f, 0.218f, 0.886f, 2.191f),
};
}  // namespace

const Variant* variants_k3s1(int* n)
{
    *n = static_cast<int>(sizeof(kTable) / sizeof(kTable[0]));
    return kTable;
}

}  // namespace conv
}  // namespace mlvc_hip
