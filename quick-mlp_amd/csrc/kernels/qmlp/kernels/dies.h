#pragma once
// Also included by the host.

namespace qmlp { namespace kernel {

/** Dies of the chip, each with an L2 of its own; workgroups go to them in turn. */
constexpr int DIES = 8;

}}
