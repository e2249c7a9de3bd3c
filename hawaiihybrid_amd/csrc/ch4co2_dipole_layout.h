// The CH4-CO2 dipole expansion laid out in (l_a, l_b) blocks for the dipole pass (hh_ch4co2.hip), on the host.
#pragma once
#include <algorithm>
#include <cstring>
#include <map>
#include <set>
#include <utility>
#include <vector>

#include "ch4co2_dipole_tables.h"

namespace hh {

// One block: its basis functions are rows [pos, pos + nb) of the radial table; the quads of component
// c are [quad[c], quad[c + 1]), the coefficients of quad q the 4 nb values from coef0 + 4 nb (q -
// quad[0]), function-major.
struct DipBlock {
    int nb, pos, coef0, pad;
    int quad[4];
};

// The expansion as a table T (Ch4Co2DipTables of the dipole pass); false, with t unfinished, when it does not fit
// T's bounds: more blocks, quads or coefficients than T holds, or a block of more functions than the pass has
// an instance for.
template <typename T>
bool fill_ch4co2_tables(T& t)
{
    using P = typename T::Real;
    // l of an X index (l^2 ..) and of a Y index (even l: l (l - 1) / 2 ..)
    auto la = [](int x) { int l = 0; while ((l + 1) * (l + 1) <= x) ++l; return l; };
    auto lb = [](int y) { int l = 0; while ((l + 2) * (l + 1) / 2 <= y) l += 2; return l; };
    struct Host {
        std::vector<int> fn;                        // basis functions
        std::vector<std::pair<int, int>> prod[3];   // products (x, y) of each component
        long cost = 0;
    };
    std::map<std::pair<int, int>, Host> blocks;
    for (int b = 0; b < HH_CH4CO2_NB; ++b)
        if (HH_CH4CO2_START[b][3] > HH_CH4CO2_START[b][0]) {
            const unsigned xy = HH_CH4CO2_XY[HH_CH4CO2_START[b][0]];
            blocks[{la(xy & 0xff), lb(xy >> 8)}].fn.push_back(b);
        }
    std::vector<Host*> order;
    for (auto& kv : blocks) {
        Host& h = kv.second;
        h.cost = 24 + 12 * (long)h.fn.size();
        for (int c = 0; c < 3; ++c) {
            std::set<std::pair<int, int>> used;
            for (int b : h.fn)
                for (int e = HH_CH4CO2_START[b][c]; e < HH_CH4CO2_START[b][c + 1]; ++e)
                    used.insert({(int)(HH_CH4CO2_XY[e] & 0xff), (int)(HH_CH4CO2_XY[e] >> 8)});
            h.prod[c].assign(used.begin(), used.end());
            h.cost += (long)(h.prod[c].size() + 3) / 4 * (8 + 4 * (long)h.fn.size());
        }
        order.push_back(&h);
    }
    // blocks to wavefronts: the costliest first, each to the least loaded wavefront
    std::stable_sort(order.begin(), order.end(), [](const Host* a, const Host* b) { return a->cost > b->cost; });
    constexpr int waves = T::kWaves;
    std::vector<Host*> share[waves];
    long load[waves] = {};
    for (Host* h : order) {
        const int w = (int)(std::min_element(load, load + waves) - load);
        share[w].push_back(h);
        load[w] += h->cost;
    }
    std::memset(&t, 0, sizeof t);
    int nblk = 0, pos = 0, quad = 0, coef = 0;
    for (int w = 0; w < waves; ++w) {
        t.wave0[w] = nblk;
        for (const Host* h : share[w]) {
            const int nb = (int)h->fn.size();
            if (nblk == T::kBlocks || nb > T::kMaxNB) return false;
            DipBlock& bl = t.block[nblk++];
            bl.nb = nb;
            bl.pos = pos;
            bl.coef0 = coef;
            for (int j = 0; j < nb; ++j, ++pos) {
                const int b = h->fn[j];
                for (int k = 0; k < HH_CH4CO2_NINT; ++k)
                    for (int i = 0; i < 4; ++i) t.radial[k][pos][i] = (P)HH_CH4CO2_RADIAL[k][b][i];
                for (int i = 0; i < 3; ++i) t.radial[HH_CH4CO2_NINT][pos][i] = (P)HH_CH4CO2_TAIL[b][i];
            }
            for (int c = 0; c < 3; ++c) {
                bl.quad[c] = quad;
                for (size_t p0 = 0; p0 < h->prod[c].size(); p0 += 4, ++quad, coef += 4 * nb) {
                    if (quad == T::kQuads || coef + 4 * nb > T::kCoefs) return false;
                    for (int u = 0; u < 4; ++u) {
                        if (p0 + u >= h->prod[c].size()) continue;   // padded: coefficients 0
                        const std::pair<int, int> xy = h->prod[c][p0 + u];
                        t.xy[quad][u] = (unsigned)xy.first | (unsigned)xy.second << 16;
                        for (int j = 0; j < nb; ++j) {
                            const int b = h->fn[j];
                            for (int e = HH_CH4CO2_START[b][c]; e < HH_CH4CO2_START[b][c + 1]; ++e)
                                if ((int)(HH_CH4CO2_XY[e] & 0xff) == xy.first && (int)(HH_CH4CO2_XY[e] >> 8) == xy.second)
                                    t.coef[coef + 4 * j + u] += (P)HH_CH4CO2_COEF[e];
                        }
                    }
                }
            }
            bl.quad[3] = quad;
        }
    }
    t.wave0[waves] = nblk;
    for (int k = 0; k < HH_CH4CO2_NINT; ++k) {
        t.bounds[k] = HH_CH4CO2_BOUNDS[k];
        t.centre[k] = HH_CH4CO2_CENTRE[k];
    }
    return true;
}

}  // namespace hh
