"""Which kernel the weight gradients of a call go to (csrc/layer.hip, csrc/wgrad_wide.hip), by the workspace that they ask for: no GPU needed."""
import pytest


def small_tile_bytes(sizes, T):
    """Workspace of the 128 x 128 tiles: parts of T until 400 workgroups run, none below 128 rows."""
    tiles = sum(-(-s[0] // 128) * -(-s[1] // 128) for s in sizes)
    parts = 1
    while parts < 8 and tiles * parts < 400 and T // (2 * parts) >= 128:
        parts *= 2
    return parts * tiles * 128 * 128 * 4


def workspace(pkg, sizes, T, pitch=0, dtype=1):
    L = pkg._lib
    jobs = (L.WgradJob * len(sizes))()
    for j, (M, N, kept, at, gap) in zip(jobs, sizes):
        j.p = j.q = j.out = 256
        j.ldp, j.ldq, j.rows, j.cols, j.keep_cols, j.gap_at, j.gap = max(M, pitch), N, M, N, kept, at, gap
    return L.load().mpa_wgrad_workspace_bytes(jobs, len(sizes), T, dtype)


@pytest.mark.parametrize("pitch,wide", [(0, True), ((1 << 25) - 8, True), (1 << 25, False)])
def test_a_slice_of_a_wide_tile_is_below_2_gb(pkg, pitch, wide):
    """32 rows of a pitch of 2^25 are 2^31 bytes, where the offset stands that the columns beyond a narrow tile have."""
    sizes = [(3072, 768, 768, 0, 0), (96, 1536, 1536, 48, 16)]
    assert (workspace(pkg, sizes, 8000, pitch) != small_tile_bytes(sizes, 8000)) == wide
