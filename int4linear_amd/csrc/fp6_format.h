// The converted (FP6) form of an operand, shared by the converter and the kernels that read it:
// [tile of 256 rows][stage of 128 k][k-fragment of 64 k][row fragment of 32 rows] x 1536 bytes, a
// fragment being 64 MFMA lanes x 16 bytes followed by 64 lanes x 8 bytes.  (Two fragments as
// three pieces of 16 bytes per lane, so that every access is 16 bytes wide, was built and measured:
// the small-grid kernel gains 0-3 %, the large one loses 3 %, because its reads come in fewer,
// larger bursts.)
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace int4linear {

constexpr int kTileRows = 256;                        // rows of either operand per tile
constexpr int kFragRows = 32;                         // rows of one MFMA operand
constexpr int kFragK = 64;                            // k of one MFMA
constexpr int kFragBytes = 64 * 24;                   // 64 lanes x 192 bits
constexpr int kFragLoBytes = 64 * 16;                 // the 16-byte parts come first
constexpr int kStageK = 128;                          // k per pipeline stage
constexpr int kFragsK = kStageK / kFragK;             // 2
constexpr int kFragsRows = kTileRows / kFragRows;     // 8
constexpr int kUnitBytes = kFragsRows * kFragBytes;   // 12 KiB: 64 k of a tile
constexpr int kOperandStageBytes = kFragsK * kUnitBytes;  // 24 KiB
constexpr float kUnscale = 64.f;                      // the codes are n/8: a product is n*m/64

}  // namespace int4linear
