#define MHD_T double
#include "k_rowpair.inc"
