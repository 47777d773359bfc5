// Register-direct transforms of the lengths 300..415.
#define DNSP_RG_NAME rg_ops_5
#define DNSP_RG_LO 300
#define DNSP_RG_HI 416
#include "poisson_reg_inst.h"
