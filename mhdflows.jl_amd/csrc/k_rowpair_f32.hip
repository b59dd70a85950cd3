#define MHD_T float
#include "k_rowpair.inc"
