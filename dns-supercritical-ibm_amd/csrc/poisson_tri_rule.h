// Instantiates the rule-shaped tridiagonal kernels (part_shape) of one spectrum
// and arithmetic type and layout; poisson_tri_rule_<i>.hip set DNSP_RULE_T,
// DNSP_RULE_AR and DNSP_RULE_MM (several files, so that they compile side by side).
#include <utility>

#include "poisson_ct.h"
#include "poisson_ct_launch.h"

namespace dnsp {

namespace {

template <int P, int M, int MR, typename T, typename Ar, bool MM>
void rule_launch(const PartArgs<T>& a, hipStream_t st) {
    const long plane = (long)a.nx * a.nz;
    // every group and the group of modes 1..M-1; or the listed ones
    const int ngroups = a.glist ? a.nlist / (M == 32 ? 2 : 1) : (int)((plane + M - 1) / M) + 1;
    if (ngroups <= 0) return;
    kt_tri_part<MR, P, M, T, 1, false, Ar, MM><<<ngroups, M * P, 3 * sizeof(Ar) * MR * P, st>>>(
        a.S, a.ax, a.az, a.bands, a.nx, a.ny, plane, a.pcr_min, a.msum, a.pbar, a.inv_nxnz, a.glist, a.nz, a.So, a.at);
}

// chunk counts and their row ranges, from part_shape's bounds
template <int P, int M, int LO, typename T, typename Ar, bool MM, int... I>
void rule_rows(const PartArgs<T>& a, int mr, hipStream_t st, std::integer_sequence<int, I...>) {
    using Fn = void (*)(const PartArgs<T>&, hipStream_t);
    static const Fn t[sizeof...(I)] = {rule_launch<P, M, LO + I, T, Ar, MM>...};
    t[mr - LO](a, st);
}

}  // namespace

template <typename T, typename Ar, bool MM>
void part_launch_rule(const PartArgs<T>& a, hipStream_t st) {
    constexpr bool F = sizeof(T) == 4;
    const PartShape s = part_shape(a.ny, F);
    static_assert(part_shape(2, F).MR == 2 && part_shape(48, F).MR == 12, "P 4: 2..12 rows");
    static_assert(part_shape(49, F).MR == 7 && part_shape(128, F).MR == 16, "P 8: 7..16 rows");
    static_assert(part_shape(129, F).MR == 9 && part_shape(512, F).MR == 32, "P 16: 9..32 rows");
    static_assert(part_shape(513, F).MR == 17 && part_shape(1024, F).MR == 32, "P 32: 17..32 rows");
    constexpr int M = part_shape(2, F).M, M32 = part_shape(1024, F).M;
    if (s.P == 4) rule_rows<4, M, 2, T, Ar, MM>(a, s.MR, st, std::make_integer_sequence<int, 11>{});
    else if (s.P == 8) rule_rows<8, M, 7, T, Ar, MM>(a, s.MR, st, std::make_integer_sequence<int, 10>{});
    else if (s.P == 16) rule_rows<16, M, 9, T, Ar, MM>(a, s.MR, st, std::make_integer_sequence<int, 24>{});
    else rule_rows<32, M32, 17, T, Ar, MM>(a, s.MR, st, std::make_integer_sequence<int, 16>{});
}

template void part_launch_rule<DNSP_RULE_T, DNSP_RULE_AR, DNSP_RULE_MM>(
    const PartArgs<DNSP_RULE_T>&, hipStream_t);

}  // namespace dnsp
