// LDS layout of the filter kernel's blocks, shared by the kernel, its launch and the
// layout test (no HIP types).
#pragma once

namespace r2 {
namespace filter_lds {

constexpr int kRow = 68;    // row of one value over a batch's hits: 16-byte aligned, rows 4 banks apart
constexpr int kWaves = 4;   // waves per 256-thread block
constexpr int kVals = 17;   // per-ray sums: S6, diffuse3, specular3, normal3, ior, distance
constexpr int kGroup = 16;  // voxels of a wave's density pass, four lanes each
constexpr int kTsFloats = 1024;  // clip distances a wave's group may hold (kGroup * 64; a voxel has up to 1000)
constexpr int kStage = 32;  // candidate triangles staged at a time (9 float4 each)
constexpr int kSumRow = 19;  // per voxel: the kVals sums, the hit count; odd, so that rows fall on distinct banks
static_assert(kStage * 9 * 4 <= kVals * kRow, "the staged triangles share the space of the per-hit values");
static_assert(kTsFloats <= kVals * kRow, "so do the exp terms of the density iteration");

// clip distances kept per voxel for n rays
constexpr int ts_cap(int n_samples) { return (n_samples + 63) / 64 * 64; }
// voxels that a wave may take together, by the clip distances it can hold
constexpr int max_group(int cap) {
  return kTsFloats / cap < 1 ? 1 : (kTsFloats / cap < kGroup ? kTsFloats / cap : kGroup);
}
// floats of a wave: [kVals][kRow] values, [group][cap] clip distances, [group][kSumRow]
// sums.  A whole number of 16-byte units: the values are read and written by float4,
// and kSumRow is odd.
constexpr int wave_floats(int group, int cap) { return (kVals * kRow + group * (cap + kSumRow) + 3) & ~3; }

}  // namespace filter_lds
}  // namespace r2
