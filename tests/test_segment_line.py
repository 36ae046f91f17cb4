"""Which backward scans of short sequences are cut into equal segments (csrc/sscan_bwd.hip: even_segments), by the workspace that they ask for: no
GPU needed."""
import ctypes

import pytest


def cut(pkg, batch, tiles, dim, states):
    L = pkg._lib
    s = L.SscanShape()
    s.batch, s.seqlen, s.dim, s.dstate = batch, 16 * tiles, dim, states
    by_rule = L.load().mpa_sscan_bwd_workspace_bytes(ctypes.byref(s))
    s.plan_segments = 1
    return by_rule != L.load().mpa_sscan_bwd_workspace_bytes(ctypes.byref(s))


# (in segments, a pass by which the host is the slower one took 1.02 to 1.09 of its time at 28 to 30 tiles, in two of them 0.95 to 1.07 at 25)
@pytest.mark.parametrize("batch,dim,states,first", [(2, 500, 16, 32), (1, 64, 16, 32), (85, 64, 16, 32), (86, 64, 16, 28), (2, 500, 32, 16), (1, 800, 64, 8),
                                                    (1, 64, 80, 7), (1, 64, 256, 7)])
def test_line(pkg, batch, dim, states, first):
    assert not cut(pkg, batch, first - 1, dim, states) and cut(pkg, batch, first, dim, states)


def segments(pkg, batch, tiles, dim):
    """Of the plan: the number that asks for the same workspace when it is pinned."""
    L = pkg._lib
    s = L.SscanShape()
    s.batch, s.seqlen, s.dim, s.dstate = batch, 16 * tiles, dim, 16
    by_rule, found = L.load().mpa_sscan_bwd_workspace_bytes(ctypes.byref(s)), []
    for n in range(1, 65):
        s.plan_segments = n
        if L.load().mpa_sscan_bwd_workspace_bytes(ctypes.byref(s)) == by_rule:
            found.append(n)
    return found


# (4 x 4096 x 40 in 64 segments of four tiles took 1.09 of the time that 32 take)
@pytest.mark.parametrize("batch,dim,tiles,want", [(4, 40, 256, 32), (3, 64, 186, 31), (1, 64, 96, 32), (1, 64, 95, 32), (1, 64, 320, 40), (1, 32, 1024, 64),
                                                  (16, 64, 256, 16), (1, 64, 33, 11)])
def test_many_segments_are_long(pkg, batch, dim, tiles, want):
    assert want in segments(pkg, batch, tiles, dim)
