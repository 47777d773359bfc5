// Register-direct transforms of the lengths 16..44.
#define DNSP_RG_NAME rg_ops_0
#define DNSP_RG_LO 16
#define DNSP_RG_HI 45
#include "poisson_reg_inst.h"
