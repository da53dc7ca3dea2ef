// Blocks of consecutive channels: the arithmetic by which the kernels cut a
// row of C channels (constexpr, so host and device code share it).
#pragma once

namespace channel_blocks {

// Most channels that one pass of a transpose stages in LDS.
constexpr int kTileChannels = 128;

// Channels per transpose pass: at most kTileChannels, the passes about equal
// and multiples of 8.  (The last pass may be left with any width from 1.)
constexpr int tile_channels(int C) {
  const int passes = (C + kTileChannels - 1) / kTileChannels;
  const int per = ((C + passes - 1) / passes + 7) / 8 * 8;
  return C < per ? C : per;
}

// Most channels that a block of the planar transpose stages in LDS, and the
// channels per block of C: about equal and multiples of 4.  (The last one may
// be left with any width from 1.)
constexpr int kPlanarChannels = 128;

constexpr int planar_blocks(int C) { return (C + kPlanarChannels - 1) / kPlanarChannels; }

constexpr int planar_channels(int C) {
  const int per = ((C + planar_blocks(C) - 1) / planar_blocks(C) + 3) / 4 * 4;
  return C < per ? C : per;
}

// First channel of the block whose nominal first channel is c (< C).  A block
// is moved as pieces of `piece` channels, the last of them ending at the
// block's end, so no block may be narrower than a piece: the last one starts
// early enough to hold one.  What it then shares with the block before it is
// moved twice, the same values.  C >= piece.
constexpr int first_channel(int C, int piece, int c) {
  return c < C - piece ? c : C - piece;
}

}  // namespace channel_blocks
