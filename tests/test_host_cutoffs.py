"""The neighbour cutoff of every pair code (nbor_setup.f): looked for over
classes of bead pairs, it is the one found over every pair of the first chains
of the species, bit for bit -- each code's own, not only the largest, from
which the cell grid follows.  Chains of 4, 5 and 6 residues, where the classes
of far residues begin; three species; the build flags; beads bonded at the
start."""
import os
import subprocess

import pytest

import pdmd

CSRC = os.path.join(pdmd.PKG_DIR, "csrc")

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include "pdmd_host.h"
using namespace pdmd;

// the cutoffs from every pair of beads: of each species' first chain, and of
// the first chains of two species
static void every_pair(const Params& p, const Topology& t, const std::vector<int>& ident, double rlsq[51]) {
    double sig[51] = {0.0}, all = 0.0;
    std::vector<int> firsts;
    for (int c = 0; c < (int)t.chain_len.size(); ++c) {
        bool seen = false;
        for (int f : firsts) seen = seen || t.species[f] == t.species[c];
        if (!seen) firsts.push_back(c);
    }
    for (size_t a = 0; a < firsts.size(); ++a)
        for (size_t b = a; b < firsts.size(); ++b)
            for (int i = t.chain_start[firsts[a]]; i < t.chain_start[firsts[a]] + 4 * t.chain_len[firsts[a]]; ++i)
                for (int j = t.chain_start[firsts[b]]; j < t.chain_start[firsts[b]] + 4 * t.chain_len[firsts[b]]; ++j) {
                    if (j <= i) continue;
                    const int code = static_code(t, j, i), x = ident[i], y = ident[j];
                    double s = 0.0;
                    if (code <= 3) s = a == b ? p.sigma_2b[x][y] : p.sigma_2b[y][x];
                    else if (code == 15) s = 0.5 * (p.welldia[x] + p.welldia[y]);
                    else if (code == 16) s = p.wel[x][y] / p.boxl_orig;
                    sig[code] = std::max(sig[code], s);
                }
    for (int k = 0; k <= 26; ++k) all = std::max(all, sig[k]);
    double shoulder = 0.0;
    for (int i = 1; i <= 4; ++i)
        for (int j = 1; j <= 4; ++j)
            if (i != 3 || j != 3) shoulder = std::max(shoulder, p.sigma[i] + p.sigma[j]);
    for (int k = 40; k <= 50; ++k) {
        sig[k] = 0.5 * shoulder;
        all = std::max(all, sig[k]);
    }
    for (int k = 0; k <= 50; ++k) {
        const double v = (kRlConst - 1) * all + sig[k];
        rlsq[k] = k >= 1 && sig[k] != 0.0 ? v * v : 0.0;
    }
}

int main(int argc, char** argv) {  // parameter folder, flags, seed, then length:species of each chain
    const int flags = std::atoi(argv[2]), seed = std::atoi(argv[3]);
    std::vector<int> len, species;
    for (int k = 4; k < argc; ++k) {
        int L, s;
        if (std::sscanf(argv[k], "%d:%d", &L, &s) != 2) return 2;
        len.push_back(L);
        species.push_back(s);
    }
    Params p;
    std::string err;
    if (!load_params(p, argv[1], err)) return 3;
    // sequences and hydrophobic flags, alike for the chains of a species
    uint64_t r = 1000u * (unsigned)seed;
    auto draw = [&](int n) { return (int)(splitmix64(r++) % (unsigned)n); };
    std::vector<int> restype, hp;
    for (size_t c = 0; c < len.size(); ++c) {
        size_t same = 0;
        while (species[same] != species[c]) ++same;
        size_t at = 0;
        for (size_t q = 0; q < same; ++q) at += len[q];
        for (int k = 0; k < len[c]; ++k) {
            restype.push_back(same < c ? restype[at + k] : 9 + draw(20));
            hp.push_back(same < c ? hp[at + k] : draw(2));
        }
    }
    scale_params(p, 120.0);
    Topology t;
    t.no_hbs = flags & 1;
    t.no_h = flags & 2;
    t.chaptype2 = flags & 4;
    t.build(len, species, restype, hp);
    std::vector<int> ident = t.ident0;
    for (int b = 0; b < t.N; ++b)
        if ((ident[b] == 1 || ident[b] == 4) && draw(3) == 0) ident[b] += 4;
    Cutoffs c;
    nbor_setup(p, t, ident, c);
    double want[51];
    every_pair(p, t, ident, want);
    int bad = 0, codes = 0;
    for (int k = 0; k <= 50; ++k) {
        codes += want[k] > 0.0;
        if (c.rlsq[k] != want[k]) {
            std::printf("code %d: %.17g, over every pair %.17g\n", k, c.rlsq[k], want[k]);
            bad = 1;
        }
    }
    std::printf("%d codes with a cutoff\n", codes);
    return bad;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("cutoffs")
    src, exe = d / "cutoffs.cpp", d / "cutoffs"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-I", CSRC, "-o", str(exe), str(src),
                    os.path.join(CSRC, "pdmd_host.cpp")], check=True)
    return str(exe)


@pytest.mark.parametrize("flags", [0, 1, 2, 3, 4], ids=["plain", "no_hbs", "no_h", "no_hbs_no_h", "chaptype2"])
@pytest.mark.parametrize("chains", ["4:0", "5:0", "6:0", "9:0 9:0", "4:0 5:1", "32:0 6:1 6:1", "16:0 4:1 7:2"])
def test_cutoff_of_every_code(program, param_dir, chains, flags):
    if flags == 4 and chains.endswith(":2"):
        pytest.skip("one unbonded species: two of them get no wells between each other, which the cutoffs do not tell apart")
    for seed in range(1, 9):
        run = subprocess.run([program, param_dir, str(flags), str(seed), *chains.split()], capture_output=True, text=True)
        assert run.returncode == 0, f"seed {seed}: {run.stdout}{run.stderr}"
