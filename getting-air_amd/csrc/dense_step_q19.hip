// The D3Q19 step kernels.
#include "dense_step.h"

template struct lbm::DenseStep<19>;
