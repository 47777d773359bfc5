// Register-direct transforms of the lengths 560..768.
#define DNSP_RG_NAME rg_ops_7
#define DNSP_RG_LO 560
#define DNSP_RG_HI 769
#include "poisson_reg_inst.h"
