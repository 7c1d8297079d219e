// Kernel instances, part 8: 32x32-MFMA tiles (gemm_t32.h) for the row counts
// between 64 and 256, each with its split-K form.
#include "gemm_registry.h"

namespace aiter_amd {

// Why these: rows between the powers of two leave a 64- or 128-row tile half
// empty, and a wider tile moves fewer LDS bytes per product (the bound of these
// kernels) than a smaller one at the same number of workgroups.  us under
// sustained load, weights rotated: bf16 600 x 7168 x 2048 22.5 (160x128)
// against 28.9 for the best power-of-two tile, 150 x 8192 x 28672 103.6
// (160x128, split 4) / 125; A4W4 150 x 14336 x 4096 11.7 (96x128) / 15.1; A8W4
// 300 x 7168 x 16384 43.5 (96x128) / 45.4, 150 x 8192 x 28672 52.2 / 60.5.
void RegBuilder::part_mid() {
    const size_t first = reg.size();
    const Variant pre = kPre, b16r{false, false, false};
#define AA_MID(F, NAME, KA, BP, BM, BN, WMW, V)                                    \
    tile(F, BM, BN, V, launch_t32<KA, BP, BM, BN, WMW>, NAME);                     \
    tsplit(F, BM, BN, V, launch_t32<KA, BP, BM, BN, WMW, false, true>, NAME);
    AA_MID(kA16W16, "a16w16", kBf16, false, 128, 64, 2, b16r)
    AA_MID(kA16W16, "a16w16", kBf16, true, 128, 64, 2, pre)
    AA_MID(kA4W4, "a4w4", kFp4, true, 32, 128, 1, pre)
    AA_MID(kA4W4, "a4w4", kFp4, true, 128, 64, 2, pre)
    AA_MID(kA8W4, "a8w4", kFp8, true, 32, 128, 1, pre)
    AA_MID(kA8W4, "a8w4", kFp8, true, 128, 64, 2, pre)
    tsplit(kA8W4, 128, 128, pre, launch_t32<kFp8, true, 128, 128, 2, false, true>, "a8w4");
    // row counts that are no power of two: not in the kernel table (its bm are powers of two)
    const size_t unlisted = reg.size();
    AA_MID(kA16W16, "a16w16", kBf16, false, 96, 128, 1, b16r)
    AA_MID(kA16W16, "a16w16", kBf16, false, 160, 128, 1, b16r)
    AA_MID(kA16W16, "a16w16", kBf16, true, 96, 128, 1, pre)
    AA_MID(kA16W16, "a16w16", kBf16, true, 160, 128, 1, pre)
    AA_MID(kA4W4, "a4w4", kFp4, true, 96, 128, 1, pre)
    AA_MID(kA4W4, "a4w4", kFp4, true, 192, 128, 2, pre)
    AA_MID(kA8W4, "a8w4", kFp8, true, 96, 128, 1, pre)
#undef AA_MID
    // reference kernel names keep resolving as they did without these tiles
    for (size_t i = first; i < reg.size(); ++i) reg[i].by_ref = false;
    for (size_t i = unlisted; i < reg.size(); ++i) reg[i].listed = false;
}

}  // namespace aiter_amd
