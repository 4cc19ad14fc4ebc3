// Instantiations of pk_scores with B registers for 24, 30 or 32 column
// blocks, two MFMA wavefronts per query tile (one translation unit, for build
// parallelism).
#include "k_pkmfma.hpp"

dense_fn get_pk4_scores_24() { return pk_scores<24, 4>; }
dense_fn get_pk4_scores_30() { return pk_scores<30, 4>; }
dense_fn get_pk4_scores_32() { return pk_scores<32, 4>; }
