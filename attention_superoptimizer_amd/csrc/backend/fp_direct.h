// Fingerprint matmuls in one launch (fp_direct.hip): whether a product is better off there than on the
// residue planes of fp_mfma.hip, and the launch for `count` of them.
#pragma once

#include <cstdint>

namespace mi355 {

bool fp_direct_pays(int batch, int m, int n, int k);
int launch_fp_direct(uint16_t const *const *A, uint16_t const *const *B, uint16_t *const *C, int const *batch, int const *m,
                     int const *n, int const *k, int count);

}  // namespace mi355
