// Modelled time of a GEMM launch per kernel instance, the dispatch's rule for
// shapes that no tuned row covers.
//
// What bounds a tile kernel here is its workgroup's own stream of stages (128
// bytes of every row of its tile: the LDS copies and reads, then the MFMAs), so
// one workgroup's time is a line in its stages, and a launch takes as many of
// those as the fullest CU has workgroups:
//   us = call + max(per_cu * (stages * stage + wg), bytes / 6.6 TB/s, traffic / 15 TB/s)
// (skinny kernels share a CU four at a time: stages * max(stage * ceil(per_cu / 4),
// shared * per_cu) + wg * ceil(per_cu / 4) inside the max).  bytes: A, B and
// out once; traffic: the operands once per tile that reads them.  A split adds
// its f32 slices at 0.22 us per MB (written, read, summed).
//
// The constants are fits to graph-replayed timings under sustained load, weights
// rotated, on one MI355X (17 to 4096 rows, N 256 to 28672, K 512 to 28672, splits
// of 2, 4 and 8): bf16 9,300 timings over 760 shapes (the forms of a t32 tile for
// the two weight orders move the same bytes and share theirs), the MX families
// an earlier 8,200 over 977 shapes of all families.  Checked on 1,450 shapes, the dispatch's choice (modelled_choice(),
// gemm.hip) is 3.3 % (bf16), 4.2 % (A4W4) and 2.6 % (A8W4) slower on average than
// the best instance timed; the simple rule alone is 14 % (row-major bf16), 11 %
// (preshuffled), 10 % and 8 %.  2 to 5 % of the shapes run over 5 % slower than by
// the rule.
//
// bf16 has no entries up to 32 rows: there the model's choices ran 7 % (row-major)
// and 4 % (preshuffled) slower than the skinny rule on average (47 shapes each, us
// rule / model: 29 x 1328 x 7168 13.6 / 18.1, preshuffled 27 x 4960 x 2560 8.8 /
// 14.6); the MX families gain (A4W4 1 %, A8W4 4 %).
#pragma once

namespace aiter_amd {

struct GemmCost {
    const char* name;   // instance name; an f32-output form takes its bf16 form's
    float stage, shared, call, wg;
};

inline const GemmCost kGemmCosts[] = {
    {"a4w4_tile_256x256_persist", 1.21, 0, 0.5, 8.37},
    {"a4w4_tile_256x256", 1.24, 0, 0.5, 9.95},
    {"a4w4_tile_128x256_persist", 0.726, 0, 1.91, 4.48},
    {"a4w4_tile_128x256", 0.74, 0, 0.5, 6.54},
    {"a4w4_tile_256x128", 0.827, 0, 1.15, 5.68},
    {"a4w4_tile_192x128", 0.712, 0, 1.07, 4.45},
    {"a4w4_tile_128x128", 0.45, 0, 0.5, 4.17},
    {"a4w4_tile_96x128", 0.407, 0, 0.891, 3.4},
    {"a4w4_tile_192x128_splitk", 0.585, 0, 7.73, 0.01},
    {"a4w4_tile_64x128_splitk", 0.253, 0, 6.68, 0.894},
    {"a4w4_tile_32x128_splitk", 0.214, 0, 6.02, 1.26},
    {"a4w4_tile_128x64_splitk", 0.295, 0, 6.9, 0.01},
    {"a4w4_tile_64x256_splitk", 0.412, 0, 6.52, 1.26},
    {"a4w4_tile_96x128_splitk", 0.347, 0, 6.69, 0.645},
    {"a4w4_tile_128x128_splitk", 0.339, 0, 7.58, 0.211},
    {"a4w4_tile_32x128", 0.265, 0, 2.81, 1.15},
    {"a4w4_skinny_m32_alds", 0.0526, 0.0491, 3.41, 0.01},
    {"a4w4_skinny_m32", 0.116, 0.12, 3, 0.0103},
    {"a4w4_skinny_m32_n32_alds", 0.0755, 0.0739, 3.49, 0.01},
    {"a4w4_skinny_m32_n32", 0.152, 0.175, 2.06, 0.77},
    {"a4w4_tile_64x128", 0.319, 0, 1.47, 2.71},
    {"a4w4_tile_128x64", 0.329, 0, 1.41, 2.8},
    {"a4w4_tile_64x256", 0.517, 0, 0.54, 4.15},
    {"a4w4_skinny_m64_n32_alds", 0.106, 0.000198, 3.81, 0.01},
    {"a4w4_skinny_m64", 0.21, 0.202, 3.03, 0.01},
    {"a4w4_skinny_m64_n32", 0.208, 0.256, 2.64, 0.344},
    {"a8w4_tile_128x256_persist", 1.07, 0, 3.22, 4.84},
    {"a8w4_tile_128x256", 1.12, 0, 0.5, 7.71},
    {"a8w4_tile_64x256", 0.773, 0, 0.852, 3.73},
    {"a8w4_tile_64x128", 0.406, 0, 1.25, 2.97},
    {"a8w4_tile_96x128", 0.65, 0, 0.957, 3.19},
    {"a8w4_tile_128x128", 0.756, 0, 0.942, 3.74},
    {"a8w4_tile_128x64", 0.483, 0, 1.55, 2.7},
    {"a8w4_tile_64x128_splitk", 0.364, 0, 6.82, 0.159},
    {"a8w4_tile_32x128_splitk", 0.291, 0, 6.6, 0.01},
    {"a8w4_tile_128x64_splitk", 0.584, 0, 3, 2.79},
    {"a8w4_tile_64x256_splitk", 0.772, 0, 6.15, 0.01},
    {"a8w4_tile_96x128_splitk", 0.52, 0, 7.42, 0.01},
    {"a8w4_tile_128x128_splitk", 0.797, 0, 3.66, 2.13},
    {"a8w4_skinny_m32_n32_alds", 0.118, 0.12, 3.5, 0.01},
    {"a8w4_skinny_m32", 0.212, 0.199, 2.18, 0.769},
    {"a8w4_skinny_m32_n32", 0.129, 0.25, 1.94, 0.885},
    {"a8w4_tile_32x128", 0.325, 0, 1.53, 2.37},
    {"a8w4_skinny_m64", 0.338, 0.359, 2.35, 0.837},
    {"a16w16_tile_256x256_bplain_flat", 1.34, 0, 0.5, 6.97},
    {"a16w16_tile_128x256_bplain", 0.821, 0, 0.5, 4.73},
    {"a16w16_tile_160x128_bplain", 0.56, 0, 0.5, 3.61},
    {"a16w16_tile_256x128_bplain", 0.761, 0, 0.5, 4.76},
    {"a16w16_tile_128x256_splitk_bplain", 0.814, 0, 6.87, 0.01},
    {"a16w16_tile_128x128_bplain", 0.469, 0, 0.5, 2.93},
    {"a16w16_tile_256x128_splitk_bplain", 0.759, 0, 4.82, 2.02},
    {"a16w16_tile_160x128_splitk_bplain", 0.542, 0, 6.59, 0.01},
    {"a16w16_tile_64x128_splitk_bplain", 0.375, 0, 5.4, 0.177},
    {"a16w16_tile_96x128_bplain", 0.417, 0, 0.5, 2.35},
    {"a16w16_tile_128x64_splitk_bplain", 0.349, 0, 3.18, 1.99},
    {"a16w16_tile_128x128_splitk_bplain", 0.483, 0, 6.22, 0.01},
    {"a16w16_tile_256x256_bplain", 1.68, 0, 1.4, 5.43},
    {"a16w16_tile_96x128_splitk_bplain", 0.436, 0, 5.73, 0.01},
    {"a16w16_tile_64x64_splitk_bplain", 0.237, 0, 5.87, 0.01},
    {"a16w16_tile_128x64_bplain", 0.309, 0, 0.561, 2.26},
    {"a16w16_tile_64x128_bplain", 0.331, 0, 0.5, 2.16},
    {"a16w16_tile_64x64_bplain", 0.244, 0, 2.26, 0.435},
    {"a16w16_skinny_m64_n32_bplain_lds", 0.137, 0.215, 1.44, 0.523},
    {"a16w16_skinny_m64_bplain", 0.246, 0.267, 2.77, 0.01},
    {"a16w16_tile_256x256_persist", 1.26, 0, 0.5, 5.94},
    {"a16w16_tile_128x256_persist", 0.753, 0, 0.5, 3.65},
    {"a16w16_tile_128x256", 0.759, 0, 0.5, 4.49},
    {"a16w16_tile_160x128", 0.56, 0, 0.5, 3.61},
    {"a16w16_tile_256x128", 0.761, 0, 0.5, 4.76},
    {"a16w16_tile_256x256", 1.26, 0, 0.5, 7.98},
    {"a16w16_tile_128x128", 0.469, 0, 0.5, 2.93},
    {"a16w16_tile_160x128_splitk", 0.542, 0, 6.59, 0.01},
    {"a16w16_tile_96x128", 0.417, 0, 0.5, 2.35},
    {"a16w16_tile_96x128_splitk", 0.436, 0, 5.73, 0.01},
    {"a16w16_tile_64x128", 0.331, 0, 0.5, 2.16},
    {"a16w16_tile_128x64_splitk", 0.349, 0, 3.18, 1.99},
    {"a16w16_tile_128x64", 0.309, 0, 0.561, 2.26},
    {"a16w16_tile_128x128_splitk", 0.483, 0, 6.22, 0.01},
    {"a16w16_tile_64x128_splitk", 0.375, 0, 5.4, 0.177},
    {"a16w16_tile_64x64_splitk", 0.237, 0, 5.87, 0.01},
    {"a16w16_tile_64x64", 0.244, 0, 2.26, 0.435},
    {"a16w16_skinny_m64_n32_alds", 0.113, 0.192, 1.43, 0.503},
    {"a16w16_skinny_m64", 0.131, 0.195, 2.26, 0.911},
};

}  // namespace aiter_amd
