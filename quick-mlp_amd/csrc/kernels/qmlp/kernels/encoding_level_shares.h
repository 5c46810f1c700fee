#pragma once
// How EncodingLevelsKernel shares out the levels of a grid; also included by the host, which sizes its grid.

#include <qmlp/kernels/dies.h>

namespace qmlp { namespace kernel {

/** Tiles of 64 points of a level whose table takes so many bytes that a wavefront of EncodingLevelsKernel takes, such that workgroups cost
 *  the same: the L1 holds up to 32 KB of a table, and much of 256 KB (16 levels of halves, 2^20 points: a microsecond for 16^3 nodes, 4 to
 *  12 for 23^3 and 33^3, 14 to 17 for each behind). */
constexpr int encodingLevelTiles(long long tableBytes) { return tableBytes <= (32 << 10) ? 8 : tableBytes <= (256 << 10) ? 2 : 1; }

/** Wavefronts of a workgroup of EncodingLevelsKernel. */
constexpr int ENCODING_LEVEL_WAVES = 4;

/** Channels of a row that EncodingRowsKernel holds 64 of in registers and LDS (33 KB). */
constexpr int ENCODING_ROWS_MAX_CHANNELS = 128;

}}
