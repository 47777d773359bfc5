// Register-direct transforms of the lengths 208..299.
#define DNSP_RG_NAME rg_ops_4
#define DNSP_RG_LO 208
#define DNSP_RG_HI 300
#include "poisson_reg_inst.h"
