// Register-direct transforms of the lengths 45..83.
#define DNSP_RG_NAME rg_ops_1
#define DNSP_RG_LO 45
#define DNSP_RG_HI 84
#include "poisson_reg_inst.h"
