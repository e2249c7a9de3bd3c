"""The layout of the CH4-CO2 dipole expansion (ch4co2_dipole_layout.h) keeps to its table's bounds: one block, one
quad, one coefficient or one function too few is refused before anything is written past them, and the
bounds that hh_ch4co2.hip states are enough.  Compiled for the host."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hawaiihybrid_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "ch4co2_dipole_layout.h"
struct Table {
    using Real = float;
    static constexpr int kWaves = 8, kBlocks = BLOCKS, kMaxNB = MAXNB, kQuads = QUADS, kCoefs = COEFS;
    float radial[HH_CH4CO2_NINT + 1][HH_CH4CO2_NB][4];
    double bounds[HH_CH4CO2_NINT], centre[HH_CH4CO2_NINT];
    hh::DipBlock block[kBlocks];
    int wave0[kWaves + 1];
    unsigned xy[kQuads][4];
    float coef[kCoefs];
};
int main()
{
    // guards behind the table: what is written past an array in it ends in the next one, past the last one here
    struct Guarded { Table t; unsigned char guard[1 << 16]; };
    Guarded* g = static_cast<Guarded*>(std::malloc(sizeof(Guarded)));
    std::memset(g->guard, 0x5a, sizeof g->guard);
    const bool ok = hh::fill_ch4co2_tables(g->t);
    for (unsigned char c : g->guard)
        if (c != 0x5a) return 3;
    std::printf("%d\n", ok ? 1 : 0);
    return 0;
}
"""


def stated():
    s = open(os.path.join(CSRC, "hh_ch4co2.hip")).read()
    out = {k: int(re.search(rf"\b{k} = (\d+)", s).group(1)) for k in ("kBlocks", "kQuads", "kCoefs")}
    out["kMaxNB"] = int(re.search(r"\bkDipMaxNB = (\d+)", s).group(1))
    return out


def fits(tmp_path, **bounds):
    b = dict(stated(), **bounds)
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-I" + CSRC, f"-DBLOCKS={b['kBlocks']}", f"-DMAXNB={b['kMaxNB']}",
                    f"-DQUADS={b['kQuads']}", f"-DCOEFS={b['kCoefs']}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, check=True)
    return r.stdout.strip() == "1"


def test_the_stated_bounds_hold_the_expansion(tmp_path):
    assert fits(tmp_path)
    assert fits(tmp_path, kQuads=2250, kCoefs=38112)   # exactly as many as there are


@pytest.mark.parametrize("bounds", [dict(kBlocks=83), dict(kMaxNB=8), dict(kQuads=2249), dict(kCoefs=38111)])
def test_one_too_few_is_refused(tmp_path, bounds):
    assert not fits(tmp_path, **bounds)
