// Instantiates the register-direct transforms (poisson_reg.h) of the lengths
// [DNSP_RG_LO, DNSP_RG_HI) and defines their table; poisson_reg_<i>.hip set
// the bounds and the name (several files, so that they compile side by side).
#include <utility>

#include "poisson_ct.h"
#include "poisson_reg.h"

namespace dnsp {

namespace {

template <int N>
struct RgLaunch {
    static constexpr int G = rg_x_lines(N), NTX = rg_threads(G * N), NTZ = rg_threads(kRgCols * N);
    static int lines_blocks(long nlines) { return (int)((nlines + 2 * G - 1) / (2 * G)); }
    static void xfwd(const double* P, double* S, long nlines, const double2* tw, hipStream_t st) {
        kr_xfwd<N, G, NTX><<<lines_blocks(nlines), NTX, 0, st>>>(P, S, nlines, tw);
    }
    static void xbwd(const double* S, double* P, long nlines, double scale, const double2* tw, hipStream_t st) {
        kr_xbwd<N, G, NTX><<<lines_blocks(nlines), NTX, 0, st>>>(S, P, nlines, scale, tw);
    }
    static void zfwd(double* S, int nx, int ny, const double2* tw, hipStream_t st) {
        kr_zfwd<N, NTZ><<<(nx + 15) / 16 * ny, NTZ, 0, st>>>(S, nx, tw);
    }
    static void zbwd(double* S, int nx, int ny, const double2* tw, hipStream_t st) {
        kr_zbwd<N, NTZ><<<(nx + 15) / 16 * ny, NTZ, 0, st>>>(S, nx, tw);
    }
};

template <int N>
constexpr RgOps rg_ops_of() {
    if constexpr (rg_supported(N))
        return RgOps{RgLaunch<N>::xfwd, RgLaunch<N>::xbwd, RgLaunch<N>::zfwd, RgLaunch<N>::zbwd};
    else return RgOps{};
}

template <int... I>
const RgOps* rg_table(int n, std::integer_sequence<int, I...>) {
    static const RgOps t[sizeof...(I)] = {rg_ops_of<DNSP_RG_LO + I>()...};
    return &t[n - DNSP_RG_LO];
}

}  // namespace

const RgOps* DNSP_RG_NAME(int n) {
    return rg_table(n, std::make_integer_sequence<int, DNSP_RG_HI - DNSP_RG_LO>{});
}

}  // namespace dnsp
