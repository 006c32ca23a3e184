"""CPU: how the tiles of two projections in one launch are spread over workgroups, for all sizes that go together."""
import os
import subprocess

from helpers import ROOT

PROGRAM = r'''
#include "project_plan.hpp"
#include <cstdio>
#include <initializer_list>
using namespace sapa::project;

static long worst32, worst16, missed;

int main() {
    for (long B = 1; B <= 300; ++B)
        for (long low = 1; low * B <= 1024; ++low)
            // the query feature of up_factor 1 .. 4 and, for what is left, of as many tiles as go with it
            for (long high : {low, 2 * low, 3 * low + 1, 4 * low - 1, 4 * low, 16 * low, 2048 / B - low}) {
                if (high < 1 || (low + high) * B > 2048) continue;
                const long tiles[2] = {high, low}, share = 256 / B > 2 ? 256 / B : 2;
                for (int nw : {8, 12}) {
                    const Spread s = plan32(tiles, B, nw);
                    if (s.blocks[0] + s.blocks[1] > share) ++worst32;
                    for (int i = 0; i < 2; ++i) missed += s.blocks[i] * s.waves * s.per < tiles[i];
                    missed += s.waves > nw || s.waves < 1;
                }
                for (int resident : {1, 2}) {
                    const Spread s = plan16(tiles, B, resident);
                    if (s.per == 1 && (s.blocks[0] + s.blocks[1]) * B > 256 * resident) ++worst16;
                    for (int i = 0; i < 2; ++i) missed += s.blocks[i] * 4 * s.per < tiles[i];
                }
            }
    printf("%ld %ld %ld\n", worst32, worst16, missed);
}
'''


def test_a_pair_of_projections_fits_its_round(tmp_path):
    """No image has more workgroups than its share of the 256 CUs (a workgroup of each feature at least), a tile per wave
    only where all workgroups are resident, and every tile has a wave."""
    source, program = tmp_path / 'plan.cpp', tmp_path / 'plan'
    source.write_text(PROGRAM)
    subprocess.check_call(['g++', '-std=c++17', '-O1', '-I', os.path.join(ROOT, 'sapa_amd', 'csrc'), str(source), '-o', str(program)])
    assert subprocess.check_output([str(program)], text=True).split() == ['0', '0', '0']
