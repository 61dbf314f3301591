// gwn_tune.hpp - the launch shapes that the batched mode's autotuner times first.
#pragma once

#include <vector>

namespace gwn {

struct batch_shape {
    int block, chunk, blocks_per_cu, traversal;
};

// The chunk length is that of whole waves; four lanes per query for every mesh (traversal 0) have one of their
// own, so their shapes come with one chunk length each (the one that a later stage's waves take over).
inline std::vector<batch_shape> batch_shapes() {
    std::vector<batch_shape> shapes;
    for (int traversal : {0, 1})
        for (int block : {64, 128, 256})
            for (int mult : {1, 4})
                for (int bpc : {2, 4, 8})
                    if (traversal != 0 || mult == 4)
                        shapes.push_back({block, block * mult, bpc, traversal});
    return shapes;
}

} // namespace gwn
