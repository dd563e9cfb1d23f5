// Kind 8 tiles (more than 64 batch rows): rows / 16, subtiles per work-group (at most), row waves
// (times two channel halves), ring stages.
#include "bsg_rows.hpp"

namespace bsgk {

namespace {
const KernelEntry kEntries[] = {
    BSG_R(8, 2, 4, 4), BSG_R(8, 3, 4, 4), BSG_R(8, 4, 4, 4), BSG_R(8, 6, 4, 4),
};
}  // namespace

const TileTable kTilesK8 = {kEntries, (int)(sizeof kEntries / sizeof kEntries[0])};

}  // namespace bsgk
