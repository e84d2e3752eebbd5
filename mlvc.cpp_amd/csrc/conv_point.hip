// Tile variants of the 1x1 kernels over flattened pixels (conv_point.hpp).

#include "conv_point.hpp"

namespace mlvc_hip {
namespace conv {

namespace {
// Of 30 combinations of waves, tiles, passes and buffers timed on 400 1x1
// convs (32-1024 -> 32-256 channels, 0.3k-0.7M pixels), these twelve with the
// conv_mfma_kernel tiles leave 0.5% of the best time on the geometric mean.
// Small tiles with whole passes in flight for few pixels (32 pixels, 64 or 256
// channels), 128-pixel tiles of up to 128 channels for many; split convs by one
// or two m-tiles.
const Variant kTable[] = {
    costed(MLVC_VARIANT_PT(1, 4, 1, 1, 32, 1, 4), 2.326f, 0.078f, 0.395f, 0.101f),
    costed(MLVC_VARIANT_PT(2, 1, 1, 1, 64, 1, 4), 2.579f, 0.031f, 0.135f, 0.051f),
    costed(MLVC_VARIANT_PT(2, 1, 1, 1, 128, 2, 2), 2.657f, 0.0f, 0.013f, 0.058f),
    costed(MLVC_VARIANT_PT(2, 1, 1, 2, 64, 2, 4), 2.682f, 0.0f, 0.283f, 0.081f),
    costed(MLVC_VARIANT_PT(2, 2, 1, 2, 32, 1, 4), 2.284f, 0.052f, 0.788f, 0.135f),
    costed(MLVC_VARIANT_PT(3, 1, 1, 4, 32, 1, 4), 2.371f, 0.057f, 1.136f, 0.171f),
    costed(MLVC_VARIANT_PT(3, 1, 1, 4, 64, 2, 3), 2.354f, 0.0f, 1.109f, 0.179f),
    costed(MLVC_VARIANT_PT(4, 1, 1, 1, 64, 2, 4), 2.600f, 0.0f, 0.261f, 0.080f),
    costed(MLVC_VARIANT_PT(4, 1, 1, 2, 64, 1, 4), 2.425f, 0.012f, 0.582f, 0.125f),
    costed(MLVC_VARIANT_PT(4, 1, 1, 4, 64, 2, 3), 1.390f, 0.0f, 1.761f, 0.207f),
    costed(MLVC_VARIANT_PTK(1, 1), 2.828f, 0.0f, 2.207f, 0.0f),
    costed(MLVC_VARIANT_PTK(2, 1), 2.456f, 0.022f, 3.344f, 0.0f),
};
}  // namespace

const Variant* variants_point(int* n)
{
    *n = static_cast<int>(sizeof(kTable) / sizeof(kTable[0]));
    return kTable;
}

}  // namespace conv
}  // namespace mlvc_hip
