// The D2Q9 step kernels.
#include "dense_step.h"

template struct lbm::DenseStep<9>;
