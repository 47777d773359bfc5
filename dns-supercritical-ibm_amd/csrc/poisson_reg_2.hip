// Register-direct transforms of the lengths 84..139.
#define DNSP_RG_NAME rg_ops_2
#define DNSP_RG_LO 84
#define DNSP_RG_HI 140
#include "poisson_reg_inst.h"
