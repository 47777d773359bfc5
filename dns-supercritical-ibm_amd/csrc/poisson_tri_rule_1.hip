// One-pass rule-shaped tridiagonal kernels, mode-major blocks.
#define DNSP_RULE_T double
#define DNSP_RULE_AR double
#define DNSP_RULE_MM true
#include "poisson_tri_rule.h"
