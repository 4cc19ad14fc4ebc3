// Instantiations of pk_scores with B registers for up to 8 or 16 column
// blocks, two MFMA wavefronts per query tile (one translation unit, for build
// parallelism).
#include "k_pkmfma.hpp"

dense_fn get_pk4_scores_8() { return pk_scores<8, 4>; }
dense_fn get_pk4_scores_16() { return pk_scores<16, 4>; }
