// One-pass rule-shaped tridiagonal kernels, FP32 spectra and arithmetic.
#define DNSP_RULE_T float
#define DNSP_RULE_AR float
#define DNSP_RULE_MM false
#include "poisson_tri_rule.h"
