// m27q_route.h -- which small-M products take the wide kernel (m27q_wide.h).
// Host code without a HIP call, so that tests can evaluate the rule.
#pragma once

#include "../../include/m27q.h"
#include "m27q_layout.h"

namespace m27q {

// Whether the int8-MFMA kernel (m27q_mma.hip) takes a type and layout: TILED
// weights of every type, GGUF-layout Q4_K / Q5_K / Q6_K.
inline bool matmul_mfma_takes(uint32_t type, int layout) {
    return layout == M27Q_LAYOUT_TILED || type == kQ4_K || type == kQ5_K || type == kQ6_K;
}

// Whether the wide kernel is the faster one for M rows (up to 64) on `sets`
// 16-row sets of weights of K columns, on `cus` CUs.  The lines were drawn
// through 21000 products of 16 to 248320 rows, 32 to 32768 columns and M = 5 to
// 64, each timed on both sides: what they choose is 0.1% slower than the faster
// side on average, and the wide kernel more than 3% slower than the other one on
// 0.2% of them (9% at most; of 4000 further ones on 0.3%, 10% at most), where
// coarser lines (sets and M alone) had it so on 6% (89% at most).
//
// What moves the lines: the wide kernel's time is a step of the largest number
// of sets that one of its waves has, so it loses just past a step (one to 1.5
// and three to four sets per CU, and 12 to 14, a second round of workgroups); a
// K slice starts up once whatever its length (short K), and past a K of about
// 16000 the activation rows of a workgroup's step lie in too many lines.
inline bool matmul_wide_wins(uint32_t type, int layout, long long sets, int K, int M, int cus) {
    const bool gguf = layout == M27Q_LAYOUT_GGUF, q80 = type == kQ8_0;
    const long long c = cus;
    if (!matmul_mfma_takes(type, layout)) {
        // GGUF Q8_0 / IQ4_XS, against the VALU kernel, which reads whole rows
        // where this kernel's loads are narrow (us, VALU / wide): IQ4_XS 17408 x
        // 5120 at M = 3 21.9 / 34.3, Q8_0 1024 x 5120 at M = 5 39.9 / 15.8;
        // 6144 x 6144 at M = 9 85.4 / 36.0, 50000 x 2048 54.1 / 83.2; 100000 x
        // 2048 at M = 17 132.9 / 161.4.
        if (M <= 4) return false;
        if (M <= 8) return sets <= c && K >= (q80 ? 384 : 1152);
        if (M <= 16) {
            if (sets <= 2 * c) return true;
            if (sets <= 3 * c) return K >= (q80 ? 384 : 512);
            if (q80) return K >= (sets <= 4 * c ? 1024 : 2560) && sets <= 8 * c;
            return K >= (sets > 5 * c && sets <= 6 * c ? 2560 : 1280);
        }
        return M > 24 || sets <= 10 * c || K >= (sets > 20 * c ? 2304 : q80 ? 768 : 512);
    }
    // The others, against a launch of the MFMA kernel per 16 rows (us, MFMA / wide).
    if (M <= 16) return false;
    if (M > 32 || sets <= c) return true;  // Q4_K 17408 x 5120 at M = 64 86.1 / 39.3; at least 1.03x past 32 rows
    if (2 * sets < 3 * c) return false;    // Q6_K 5120 x 17408 at M = 17 45.3 / 48.3
    // M up to 24: the second launch has at most 8 rows and packs K in their place.
    const bool two = M > 24;
    const bool pair = sets <= 2 * c, past3 = sets > 3 * c && sets < 4 * c, past12 = sets > 12 * c && sets <= 14 * c;
    switch (type) {
        case kQ4_K:  // 8192 x 17408 at M = 24 40.1 / 37.4, at M = 32 47.1 / 38.1; x 2560 at M = 24 10.3 / 10.9
            if (!pair) return two || gguf || K < 4096 || !past12;  // 50000 x 5120 at M = 17 62.3 / 65.9
            if (gguf) return two ? K <= 17408 : K <= 8960 && (K <= 1024 || K >= 2304);
            return two || K <= 1024 || (K >= 7168 && K <= 12288);
        case kQ5_K:  // 6144 x 17408 at M = 17 38.3 / 47.3, x 1024 7.2 / 6.8
            if (!pair) return two || gguf || K < 4096 || !past12;
            if (gguf) return two ? K <= 17408 : K <= 9984 && (K <= 1536 || K >= 2304);
            return two ? K <= 13824 : K <= 1024 || (K >= 3584 && K <= 10240);
        case kQ6_K: {  // 8192 x 5120 at M = 17 20.9 / 18.7; GGUF rows of an odd block count start 2 bytes off a dword
            if (!gguf) return !pair || two || K <= 12288;
            const bool odd = K / 256 % 2;  // 28756 x 9984 at M = 17 117 / 134, 27960 x 8704 at M = 28 108 / 83
            if (pair) return false;
            if (past3) return K < 16384 && !(odd && (K > 5888 || (K > 512 && K < 1280)));
            return sets < 4 * c || !(odd && K > 8192 && K < 15360 && sets <= 8 * c);
        }
        case kQ8_0:  // 6144 x 2048 at M = 17 10.6 / 12.3, 10240 x 5120 33.0 / 25.8, 14336 x 1024 10.9 / 14.0
            if (pair) return two && K >= 4352;
            if (sets < 4 * c) return K >= 2560 || (K >= 1600 && !past3 && 16 * sets > 33 * c);
            return two || sets <= 12 * c || K <= 512 || K >= 1600;
        default:  // IQ4_XS 6144 x 6144 at M = 17 19.6 / 21.9, 50000 x 5120 81.1 / 93.3, 17408 x 5120 42.5 / 38.1
            if (pair) return false;
            if (past3) return K <= 896 || (two && K >= 1280);
            if (sets < 4 * c) return two || K <= 896 || K >= 3584 || 16 * sets > 33 * c;
            return two ? K <= 7168 || sets <= 12 * c : K <= (sets <= 8 * c ? 7424 : 4864);
    }
}

}  // namespace m27q
