// One-pass rule-shaped tridiagonal kernels, in place.
#define DNSP_RULE_T double
#define DNSP_RULE_AR double
#define DNSP_RULE_MM false
#include "poisson_tri_rule.h"
