// Which parameters each launch of a model brings into L2 for the launch behind it (ReefPrefetch).
#pragma once
#include <cstdint>
#include <vector>

#include "executor/model.h"
#include "reef_kernels.h"

namespace reef {
namespace executor {

// records[i]: what launch i prefetches; wgs == 0: nothing.  `storage`: device address of every storage.
// The last small operand is left for the argument block of the next launch, which only
// the caller knows.  A launch qualifies as the host of prefetching workgroups when its op knows its own
// task count (reef_entries.hip) and its last pointer slot is free.
std::vector<ReefPrefetch> plan_prefetch(const Model& model, const std::vector<void*>& storage);

}  // namespace executor
}  // namespace reef
