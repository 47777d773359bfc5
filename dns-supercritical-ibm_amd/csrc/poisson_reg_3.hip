// Register-direct transforms of the lengths 140..207.
#define DNSP_RG_NAME rg_ops_3
#define DNSP_RG_LO 140
#define DNSP_RG_HI 208
#include "poisson_reg_inst.h"
