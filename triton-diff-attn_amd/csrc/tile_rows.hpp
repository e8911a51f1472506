// The rows that one piece of a tile copy reads where the tensor ends inside the tile or in front of it.  Plain C++: a test
// compiles it by itself.
#pragma once

namespace da_abi {

// Row r of the piece reads row base + min(r, most), which is row first + r, or the tensor's last row where that lies behind it.
// `first`: the piece's first row; `last_row`: the tensor's last one (both relative to the tile, so `last_row` is negative where the
// whole tile lies past the end); the piece has `rows` rows.  Both results are the same for all lanes of a wave.
struct PieceRows { int base, most; };
constexpr PieceRows clamp_piece(int first, int last_row, int rows) {
  const int base = first < last_row ? first : last_row;
  const int room = last_row - base;
  return {base, room < rows - 1 ? room : rows - 1};
}

}  // namespace da_abi
