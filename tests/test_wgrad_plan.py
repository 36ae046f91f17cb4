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


def layer(width):
    """The four products of a layer: in_proj, out_proj, x_proj on its padded rows, dt_proj."""
    inner, rank = 2 * width, -(-width // 16)
    padded = -(-(rank + 32) // 64) * 64
    return [(2 * inner, width, width, 0, 0), (width, inner, inner, 0, 0), (padded, inner, inner, 0, 0), (inner, -(-rank // 8) * 8, rank, 0, 0)]


@pytest.mark.parametrize("width,T,wide", [(768, 8000, True), (1024, 16384, True), (640, 9000, True), (512, 8192, True),
                                          (768, 2048, False), (256, 16000, False), (128, 4096, False)])
def test_layers(pkg, width, T, wide):
    assert (workspace(pkg, layer(width), T) != small_tile_bytes(layer(width), T)) == wide


def test_sizes_that_are_checked_on_a_gpu_are_wide(pkg):
    from test_wgrad_wide_gpu import SIZES
    for T, sizes in SIZES[:4]:
        assert workspace(pkg, sizes, T) != small_tile_bytes(sizes, T)
