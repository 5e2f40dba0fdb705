// vx3h_tune.h -- the autotuner's choice among its measured candidates.
#ifndef VX3H_TUNE_H
#define VX3H_TUNE_H
#include <cstddef>
#include <vector>

#include "../../include/vx3h.h"

namespace vx3 {

// The fastest candidate; one with a workgroup size of its own only if it leads those without by
// more than two runs of one configuration differ (up to 1%).  Such a size holds for whatever the
// configuration runs later, and takes the kernels with the links of all axes at once, which choose
// their own, out of the question.
inline size_t chooseTrial(const std::vector<vx3h_tune_trial>& t) {
    size_t any = 0, free = t.size();
    for (size_t i = 0; i < t.size(); i++) {
        if (t[i].voxel_steps_per_s > t[any].voxel_steps_per_s) any = i;
        if (t[i].block_size == 0 && (free == t.size() || t[i].voxel_steps_per_s > t[free].voxel_steps_per_s)) free = i;
    }
    return free < t.size() && t[any].voxel_steps_per_s <= 1.02 * t[free].voxel_steps_per_s ? free : any;
}

}  // namespace vx3
#endif
