#pragma once
// How the slices of a grid's gradient table are shared out over workgroups (kernels/grid_gradient.h). The same definition
// is compiled by the host code, which makes the work items, and, at run time, by the device compiler: the records
// kernel zeroes what several work items of the host's add to.

namespace qmlp { namespace kernel {

/** Every level gets about this many work items of the slice kernel. */
constexpr int GRID_GRADIENT_ITEMS_PER_LEVEL = 32;

/** Work items that share out the regions of each slice of a level of so many slices. */
constexpr int gridGradientParts(int slices)
{
    return GRID_GRADIENT_ITEMS_PER_LEVEL / slices > 1 ? GRID_GRADIENT_ITEMS_PER_LEVEL / slices : 1;
}

/** Lanes of a workgroup of GridGradientExceptionsKernel. */
constexpr int GRID_GRADIENT_EXCEPTIONS_BLOCK = 256;

}} // namespace qmlp::kernel
