// Register-direct transforms of the lengths 416..559.
#define DNSP_RG_NAME rg_ops_6
#define DNSP_RG_LO 416
#define DNSP_RG_HI 560
#include "poisson_reg_inst.h"
