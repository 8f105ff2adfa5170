// The D3Q27 step kernels.
#include "dense_step.h"

template struct lbm::DenseStep<27>;
