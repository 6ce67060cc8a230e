// slab_walk.h — the columns that a wave of linear_slab_kernel reads, and the slices it takes (plain C++: the host's self-test walks them too)
#pragma once
namespace nvr {

constexpr int SLAB_WAVES = 8, SLAB_STEP = 32 * SLAB_WAVES;      // of every SLAB_STEP columns of a slice each wave multiplies 32
constexpr int SLAB_SET = 2;                                     // steps requested together

// Slices of whole sets for every wave, two of them at least: a wave then asks for no column that it does not multiply.  Others stay with linear_skinny_kernel, whose requests carry a condition: in
// this kernel, whose requests have none, a wave without a step would read behind the last slice's columns, and one with an odd number of them would ask for its last one twice.
// us, skinny / slab, such slices with the last step asked for again (4 and 20 rows): 4 slices of 256 of 12288 rows of W 9.2 / 19.0, 12.7 / 22.3; 8 of 512 of 4096 9.5 / 15.0, 13.0 / 17.3; 4 of 768
// 8.4 / 9.4, 9.9 / 10.4; 4 of 1280 13.5 / 14.8, 15.6 / 16.7.  Slices that it takes (1, 16 and 32 rows): 4 of 1024 of 4096 9.2 / 9.1, 10.3 / 10.3, 12.0 / 11.6; 4 of 1536 13.6 / 13.1, 15.5 / 15.0,
// 18.2 / 17.2; 1 of 2048 of 8192 15.0 / 14.7, 16.1 / 15.3, 18.1 / 17.2; 4 of 3072 of 4096 24.4 / 23.3, 27.5 / 26.4, 31.9 / 29.9
constexpr bool slab_takes(long kslice) { return kslice % (SLAB_SET * SLAB_STEP) == 0 && kslice >= 2 * SLAB_SET * SLAB_STEP; }
constexpr int slab_steps(int kslice) { return kslice / SLAB_STEP; }
constexpr int slab_column(int kslice, int z, int wave) { return z * kslice + wave * 32; }      // of a wave's step 0; SLAB_STEP further on the next one's

}  // namespace nvr
