// Rules on sizes that pick the N-D executor's kernels, at sizes that no test can run: nothing
// that a general kernel takes is refused because a faster one cannot.
#include <cstdio>

#include "nd_kernels.h"

static int failures = 0;
static void check(bool ok, const char *what) {
    if (ok) return;
    std::printf("FAILED: %s\n", what);
    failures++;
}

int main() {
    using ocr::nd_attention_mfma_fits;
    check(nd_attention_mfma_fits(16, 109, 8, 15), "a batch of 16 lines");
    check(nd_attention_mfma_fits(65535, 1, 1, 4) && nd_attention_mfma_fits(1, 1, 4 * 65535, 16), "largest batch and head count");
    // Left to the general kernel: offsets within an image past 2^31, more query tiles than a grid has.
    check(nd_attention_mfma_fits(1, 682, 65535, 16) && !nd_attention_mfma_fits(1, 683, 65535, 16), "values of an image");
    check(!nd_attention_mfma_fits(65535, 600000, 1, 4), "query tiles");
    check(!nd_attention_mfma_fits(1, 10, 1, 3) && !nd_attention_mfma_fits(1, 10, 1, 17), "head sizes");
    if (!failures) std::printf("all checks passed\n");
    return failures != 0;
}
