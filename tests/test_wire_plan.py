"""The host's plan of wire calls by tile, compiled from the kernels' own header (no GPU
call): a group's wires are at most a lane each whatever the device's unit count."""
import os
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
SCREENS = [(1920, 1080), (3840, 2160), (7680, 4320), (640, 360), (97, 61), (16384, 3), (3, 16384), (16384, 2000)]
MAIN = r'''
#include "%s/taichi_three_amd/csrc/wire_kernels.h"
#include <stdio.h>
#include <stdlib.h>
using namespace tina;
int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3) {
    const WireScratch w = wire_scratch(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]));
    printf("%%ld %%d %%d\n", (long)w.bytes, w.bytes ? w.room : 0, kBinBlock);
  }
  return 0;
}
'''


@pytest.fixture(scope='module')
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp('plan')
    src, exe = d / 'plan.hip', d / 'plan'
    src.write_text(MAIN % ROOT)
    subprocess.run([HIPCC, '--offload-arch=gfx950', '-O1', '-std=c++17', '-ffp-contract=off', '-Xclang', '-target-feature',
                    '-Xclang', '-packed-fp32-ops', '-o', str(exe), str(src)], check=True)

    def run(*args):
        out = subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True).stdout
        return [[int(x) for x in line.split()] for line in out.splitlines()]
    return run


@pytest.mark.parametrize('ncu', [16, 32, 64, 80, 128, 256, 304])
def test_a_group_has_a_lane_for_every_wire(plan, ncu):
    """k_wire_bin holds one wire a lane: on a device of fewer units than 256 a launch
    takes fewer wires, so that its groups stay as long as the workgroup."""
    rows = plan(*[x for W, H in SCREENS for x in (W, H, ncu)])
    assert len(rows) == len(SCREENS) and sum(r[0] > 0 for r in rows) >= 6
    for nbytes, room, lanes in rows:
        assert -(-room // ncu) <= lanes
        assert nbytes == 0 or room >= 1024
