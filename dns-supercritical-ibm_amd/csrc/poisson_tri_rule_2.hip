// One-pass rule-shaped tridiagonal kernels, FP32 spectra, FP64 arithmetic.
#define DNSP_RULE_T float
#define DNSP_RULE_AR double
#define DNSP_RULE_MM false
#include "poisson_tri_rule.h"
