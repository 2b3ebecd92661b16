// dQ and dK/dV for tensors that end inside the last block (FBSA_FLAG_RAGGED): the
// kernels of fbsa_bwd.hip with the limits on their copies, in an object of their
// own so that the two sets compile side by side.
#define FBSA_BWD_RAGGED 1
#include "fbsa_bwd.hip"
