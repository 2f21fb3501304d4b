// Lane-tile layout of a bank's stored inverse (k_mas_lanes).
//
// The dim x dim symmetric inverse (dim = 3 * bank) is cut into 8 x 8 tiles;
// tiles a >= b (block row a, block column b) are stored, a diagonal tile whole.
// Lane l = 8 ty + tx of a wave owns element (8 a + ty, 8 b + tx) of every
// stored tile, its value number a (a + 1) / 2 + b.  The values lie lane by
// lane in groups of 16 bytes (four FP32 or eight 16-bit values; one 1 KB wave
// load per group), then the few left over, padded to whole 4-byte words.
#pragma once

namespace masx
{
// values of one lane, padded to whole words
__host__ __device__ constexpr int lane_tile_count(int bank, bool f32)
{
    const int t = 3 * bank / 8, n = t * (t + 1) / 2;
    return f32 ? n : (n + 1) / 2 * 2;
}

// 4-byte words of one lane
__host__ __device__ constexpr int lane_tile_words(int bank, bool f32)
{
    return lane_tile_count(bank, f32) / (f32 ? 1 : 2);
}

// stored values of a bank
__host__ __device__ constexpr int lane_tile_values(int bank, bool f32) { return 64 * lane_tile_count(bank, f32); }

// position (in stored values) of element (i, j) of a stored tile (i / 8 >= j / 8)
__host__ __device__ constexpr int lane_tile_slot(int bank, bool f32, int i, int j)
{
    const int a = i / 8, b = j / 8, lane = 8 * (i % 8) + j % 8, s = a * (a + 1) / 2 + b;
    const int group = f32 ? 4 : 8, whole = lane_tile_count(bank, f32) / group * group;
    return s < whole ? (s / group * 64 + lane) * group + s % group
                     : 64 * whole + lane * (lane_tile_count(bank, f32) - whole) + (s - whole);
}
}  // namespace masx
