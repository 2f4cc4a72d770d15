"""CPU test of the order in which attention's tiles of queries are dealt to workgroups (tile_of_workgroup of attention_common.h, compiled for the host): every tile is dealt once; an XCD's list
starts with the longest tiles of a causal launch and goes on to ever shorter ones, and no XCD has more than a longest tile's work more than another."""
import os
import subprocess

import pytest

from metalhlo_amd import build

SOURCE = r"""
#include <cstdio>
#include "attention_common.h"
int main() {
    int heads, nqb, cus;
    while (scanf("%d %d %d", &heads, &nqb, &cus) == 3) {
        mhip::FaArgs a = {};
        a.B = 1; a.H = heads; a.nqb = nqb; a.cu_group = cus;
        for (int id = 0; id < heads * nqb; id++) {
            int t[3][2];
            mhip::tile_of_workgroup<true>(a, id, t[0][0], t[0][1]);
            mhip::tile_of_workgroup<false>(a, id, t[1][0], t[1][1]);
            mhip::tile_of_workgroup<true, false>(a, id, t[2][0], t[2][1]);
            printf("%d %d %d %d %d %d\n", t[0][0], t[0][1], t[1][0], t[1][1], t[2][0], t[2][1]);
        }
    }
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    where = tmp_path_factory.mktemp("tiles")
    source, program = where / "tiles.hip", where / "tiles"
    source.write_text(SOURCE)
    include = [a for d in (build.CSRC, os.path.join(build.ROOT, "include")) for a in ("-I", d)]
    subprocess.run([build.hipcc(), "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", *include, str(source), "-o", str(program)], check=True, capture_output=True)

    def run(heads, nqb, cus):
        out = subprocess.run([str(program)], input=f"{heads} {nqb} {cus}\n", capture_output=True, text=True, check=True).stdout
        rows = [tuple(map(int, line.split())) for line in out.splitlines()]
        return [[r[2 * k:2 * k + 2] for r in rows] for k in range(3)]
    return run


@pytest.mark.parametrize("heads", [1, 2, 3, 5, 7, 8, 9, 12, 15, 16, 20, 28, 31, 36, 77])
def test_lists(deal, heads):
    for nqb in (1, 2, 3, 8, 12, 13, 32, 47):
        for cus in (32, 5):
            orders = deal(heads, nqb, cus)
            for order in orders:
                assert len(order) == heads * nqb and set(order) == {(h, q) for h in range(heads) for q in range(nqb)}, (nqb, cus)
            work = []
            for xcd in range(8):
                mine = [q for _, q in orders[0][xcd::8]]
                # rounds of a tile a unit, every other one dealt backwards
                dealt = [q for r in range(0, len(mine), cus) for q in (mine[r:r + cus] if r // cus % 2 == 0 else mine[r:r + cus][::-1])]
                assert dealt == sorted(mine, reverse=True), (nqb, cus, xcd)
                work.append(sum(q + 1 for q in mine))
            assert max(work) - min(work) <= nqb, (nqb, cus, work)
