"""How far past the end of a line a sweep's last segment reaches: cells are found by
one wrap (csrc/gkm_sweep.hpp: wrapi), so every cell a workgroup names has to lie
below 2 nc.  On the host, for every grid, direction, tile variant, precision and
segment length that the library's own rules give (a single grid's for several
device sizes, an ensemble's for every limit it tries): the cells of the last
segment's stencils, and for FP64 the window's cells loaded ahead."""
import ctypes
import os
import re

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "..", "dns_gkm_lpt_amd", "libdnsgkm.so")


def tiles(name):
    src = open(os.path.join(HERE, "..", "dns_gkm_lpt_amd", "csrc", "gkm_kernels.hpp")).read()
    body = src[src.index(name + "[3]"):]
    v = [int(x) for x in re.findall(r"\d+", body[body.index("{"):body.index("};")])]
    return [[tuple(v[9 * d + 3 * k:9 * d + 3 * k + 3]) for k in range(3)] for d in range(3)]


def farthest(nc, CN, seg, mixed):
    """Largest cell named by the last segment's workgroups."""
    start = (nc - 1) // seg * seg
    if mixed:
        return start + seg - 1 + 3
    ahead = [start + c * CN + CN + 3 + CN - 1 for c in range(-1, seg // CN - 1)]
    return max(ahead + [start - CN - 2 + CN + 4])


@pytest.mark.parametrize("mixed", [0, 1])
def test_segments_stay_below_one_wrap(mixed):
    if not os.path.exists(LIB):
        from dns_gkm_lpt_amd import build
        build.build()
    L = ctypes.CDLL(LIB)
    seg_len = getattr(L, "_ZN3gkm13sweep_seg_lenEiiiib")
    seg_most = getattr(L, "_ZN3gkm14sweep_seg_mostEiiiib")
    tile_ok = getattr(L, "_ZN3gkm13sweep_tile_okEiii")
    tile_ok.restype = ctypes.c_bool
    shapes = tiles("kTiles" if mixed else "kTilesPair")
    bad = []
    for nc in range(16, 1025):
        for d in range(3):
            for v in range(3):
                if not tile_ok(d, v, nc):
                    continue
                CN = shapes[d][v][0]
                segs = {seg_len(d, nc, v, s, mixed) for s in (0, 32, 64, 128, 256, 512, 608, 1024)}
                segs |= {seg_most(d, nc, v, m, mixed) for m in (1 << 20, 24, 16, 12, 8, 6, 4, 3, 2, 1)}
                for seg in segs:
                    assert seg > 0 and seg % CN == 0
                    if farthest(nc, CN, seg, mixed) >= 2 * nc:
                        bad.append((nc, d, v, seg))
    assert not bad, bad
