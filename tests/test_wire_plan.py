"""The host's plan of wire calls by tile, compiled from the kernels' own header (no GPU
call): a group's wires are at most a lane each whatever the device's unit count, and
the entries of as many wires as go at a time have a count of 32 bits."""
import os
import subprocess

import numpy as np
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
  if (argc == 4 && argv[3][0] == '/') {  // wires (ax ay kx ky siz first last) from a file: tiles of each, -1: drawn
    const int tx = (atoi(argv[1]) + kWireTile - 1) / kWireTile, ty = (atoi(argv[2]) + kWireTile - 1) / kWireTile;
    FILE* f = fopen(argv[3], "rb");
    float4 w;
    int i[3];
    while (fread(&w, 16, 1, f) == 1 && fread(i, 4, 3, f) == 3) {
      long n = 0;
      const bool listed = wire_listed(w.x, w.y, w.z, w.w, i[0], 0.5f, 0.5f);
      if (listed) wire_tiles(w, i[0], i[1], i[2], 0.5f, 0.5f, tx, ty, [&](int t) { n += t >= 0 && t < tx * ty ? 1 : 1 << 30; });
      printf("%%ld\n", listed ? n : -1);
    }
    return 0;
  }
  for (int i = 1; i + 3 < argc; i += 4) {
    const int ncu = atoi(argv[i + 2]);
    const WireScratch w = wire_scratch(atoi(argv[i]), atoi(argv[i + 1]), ncu, atoi(argv[i + 3]));
    if (!w.bytes) {
      printf("0 0 0 0 0\n");
      continue;
    }
    const int per = wires_per_group(w.room, ncu);
    printf("%%ld %%d %%d %%d %%ld\n", (long)w.bytes, w.room, per - kBinBlock, (w.room + per - 1) / per,
           (long)((w.chunk_off - w.chunk_cnt) / 4 / w.ntiles));
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
    """k_wire_bin holds one wire a lane: where there are more wires than a lane each on
    every unit, there are more groups, each as long as the workgroup, and rows for them."""
    counts = (65536, 200000, 500000, 1 << 20, 3000000)
    rows = plan(*[x for W, H in SCREENS for n in counts for x in (W, H, ncu, n)])
    assert len(rows) == len(SCREENS) * len(counts) and sum(r[0] > 0 for r in rows) >= 30
    for (nbytes, room, over, groups, tables), n, (W, H) in zip(rows, counts * len(SCREENS),
                                                               [s for s in SCREENS for _ in counts]):
        assert over <= 0 and groups <= tables
        # one launch takes the whole call, up to 2^20 wires and what 32 bits of entries allow
        assert nbytes == 0 or room >= min(n, 1 << 20) or room >= 2 ** 32 // (4 * (-(-W // 32) + -(-H // 32) + 5))


@pytest.mark.parametrize('W,H', SCREENS)
def test_entries_keep_a_count_of_32_bits(plan, tmp_path, W, H):
    """Wires that start on the screen or beside it and end up to 2^31 pixels away, along
    both axes and at slopes near one: a listed wire has at most three entries a tile of
    its major axis, so that the room's wires together stay below 2^32 of them."""
    tx, ty = -(-W // 32), -(-H // 32)
    (nbytes, room, *_), = plan(W, H, 256, 1 << 20)
    rng = np.random.default_rng(3)
    n = 600
    w = np.zeros(n, dtype=[('p', '<f4', 4), ('i', '<i4', 3)])
    siz = np.exp(rng.uniform(np.log(1.0), np.log(2.0 ** 31 - 1), n))
    siz[:60], siz[60:120] = 2.0 ** 31 - 1, 7.9e6
    start = rng.uniform(-0.1, 1.1, (n, 2)) * (W, H)
    minor = np.where(rng.random(n) < 0.5, rng.choice([-1.0, 0.0, 1.0], n), rng.uniform(-1, 1, n))
    major = rng.choice([-1.0, 1.0], n)
    xm = np.abs(minor) == 1.0
    xm |= rng.random(n) < 0.5
    w['p'][:, :2] = start
    w['p'][:, 2], w['p'][:, 3] = np.where(xm, major, minor), np.where(xm, minor, major)
    w['i'][:, 0] = siz
    # the walked steps, with the set-up's margin on the major axis
    a, res = np.where(xm, start[:, 0], start[:, 1]), np.where(xm, W, H)
    err = 2 + (np.abs(a) + siz + 1 + res) * 1e-6
    lo = np.clip(np.where(major > 0, -a - err, a - res - err), 0, siz)
    hi = np.clip(np.where(major > 0, res - a + err, a + err), 0, siz)
    w['i'][:, 1], w['i'][:, 2] = np.ceil(lo), np.floor(hi)
    (tmp_path / 'wires').write_bytes(w.tobytes())
    tiles = np.array(plan(W, H, tmp_path / 'wires'))[:, 0]
    assert len(tiles) == n and (tiles >= 0).sum() > n / 3 and (tiles < 0).sum() >= 60
    assert tiles.max() <= 3 * max(tx, ty)
    assert nbytes == 0 or room * int(3 * max(tx, ty)) < 2 ** 32
