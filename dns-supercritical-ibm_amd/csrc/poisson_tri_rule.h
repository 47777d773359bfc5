// Instantiates the rule-shaped tridiagonal kernels (part_shape) of one chunk
// form and layout; poisson_tri_rule_<i>.hip set DNSP_RULE_TP and DNSP_RULE_MM
// (several files, so that they compile side by side).
#include <utility>

#include "poisson_ct.h"
#include "poisson_ct_launch.h"

namespace dnsp {

namespace {

template <int P, int M, int MR, bool TP, bool MM>
void rule_launch(const PartArgs& a, hipStream_t st) {
    const long plane = (long)a.nx * a.nz;
    const int ngroups = (int)((plane + M - 1) / M) + 1;  // and the group of modes 1..M-1
    kt_tri_part<MR, P, M, double, 1, TP, double, MM><<<ngroups, M * P, 3 * sizeof(double) * MR * P, st>>>(
        a.S, a.ax, a.az, a.bands, a.nx, a.ny, plane, a.pcr_min, a.msum, a.pbar, a.inv_nxnz, nullptr, a.nz, a.So);
}

// chunk counts and their row ranges, from part_shape's bounds
template <int P, int M, int LO, bool TP, bool MM, int... I>
void rule_rows(const PartArgs& a, int mr, hipStream_t st, std::integer_sequence<int, I...>) {
    using Fn = void (*)(const PartArgs&, hipStream_t);
    static const Fn t[sizeof...(I)] = {rule_launch<P, M, LO + I, TP, MM>...};
    t[mr - LO](a, st);
}

}  // namespace

template <bool TP, bool MM>
void part_launch_rule(const PartArgs& a, hipStream_t st) {
    const PartShape s = part_shape(a.ny);
    static_assert(part_shape(2).MR == 2 && part_shape(48).MR == 12, "P 4: 2..12 rows");
    static_assert(part_shape(49).MR == 7 && part_shape(128).MR == 16, "P 8: 7..16 rows");
    static_assert(part_shape(129).MR == 9 && part_shape(512).MR == 32, "P 16: 9..32 rows");
    static_assert(part_shape(513).MR == 17 && part_shape(1024).MR == 32, "P 32: 17..32 rows");
    if (s.P == 4) rule_rows<4, 16, 2, TP, MM>(a, s.MR, st, std::make_integer_sequence<int, 11>{});
    else if (s.P == 8) rule_rows<8, 16, 7, TP, MM>(a, s.MR, st, std::make_integer_sequence<int, 10>{});
    else if (s.P == 16) rule_rows<16, 16, 9, TP, MM>(a, s.MR, st, std::make_integer_sequence<int, 24>{});
    else rule_rows<32, 8, 17, TP, MM>(a, s.MR, st, std::make_integer_sequence<int, 16>{});
}

template void part_launch_rule<DNSP_RULE_TP, DNSP_RULE_MM>(const PartArgs&, hipStream_t);

}  // namespace dnsp
