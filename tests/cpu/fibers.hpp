// Runs a kernel's workgroups one after another, the threads of a workgroup as
// fibers: each runs to its next barrier before another one does, in the order
// that `descending` chooses.  A result that depends on the order within a
// workgroup is a race between two of its barriers.
#pragma once

#include <functional>

namespace fibers {

extern bool descending;
void launch(unsigned blocks, unsigned threads, const std::function<void()>& kernel);

}  // namespace fibers
