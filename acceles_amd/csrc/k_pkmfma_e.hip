// Instantiations of pk_scores with B registers for up to 30 column blocks
// (one translation unit each, for build parallelism).
#include "k_pkmfma.hpp"

dense_fn get_pk_scores_30() { return pk_scores<30, 0>; }
