// Dispatch of the register-direct transforms over the files that hold them.
#include "poisson_ct_launch.h"

namespace dnsp {

const RgOps* rg_ops_0(int n);
const RgOps* rg_ops_1(int n);
const RgOps* rg_ops_2(int n);
const RgOps* rg_ops_3(int n);
const RgOps* rg_ops_4(int n);
const RgOps* rg_ops_5(int n);
const RgOps* rg_ops_6(int n);
const RgOps* rg_ops_7(int n);

const RgOps* rg_ops(int n) {
    if (!rg_supported(n)) return nullptr;
    if (n < 45) return rg_ops_0(n);
    if (n < 84) return rg_ops_1(n);
    if (n < 140) return rg_ops_2(n);
    if (n < 208) return rg_ops_3(n);
    if (n < 300) return rg_ops_4(n);
    if (n < 416) return rg_ops_5(n);
    if (n < 560) return rg_ops_6(n);
    return rg_ops_7(n);
}

}  // namespace dnsp
