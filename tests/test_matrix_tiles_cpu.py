"""Which tile a product of more than 48 rows takes on a device of 256 compute units (no GPU: the rule alone)."""
import pytest

from ternaryllm_amd import _lib

TILES = ["shared 32x32", "shared 32x64", "shared 64x64", "small", "wide", "halves", "groups", "flat", "tall"]   # in the order of tl_matrix_tile's results


def tile_of(M, K, N, dtype, two=False, planes=1, units=256):
    rc = _lib.lib().tl_matrix_tile(M, N, K, planes, _lib.TL_F32 if dtype == "fp32" else _lib.TL_F16, int(two), units)
    _lib.check(min(rc, 0))
    return TILES[rc]


# The sides of each line at which both tiles were timed: the tile that was the faster one there (us, the faster / the other).
@pytest.mark.parametrize("M,K,N,dtype,two,tile", [
    (64, 64, 4096, "fp16", False, "shared 32x32"),      # 3.6 / 3.6 small
    (64, 4096, 4096, "fp16", False, "shared 32x32"),    # 6.6 / 8.1 shared 32x64
    (128, 64, 4096, "fp16", False, "small"),            # 3.6 / 3.9 shared 32x64
    (128, 256, 4096, "fp16", False, "small"),           # 4.2 / 4.7 shared 32x64
    (200, 256, 2048, "fp16", False, "small"),           # 4.1 / 4.7 shared 32x64
    (128, 512, 4096, "fp16", False, "shared 32x64"),    # 4.7 / 4.8 small
    (256, 256, 4096, "fp16", False, "small"),           # 4.3 / 5.3 shared 32x64
    (256, 768, 4096, "fp16", False, "small"),           # 5.8 / 6.1 shared 32x64
    (256, 1024, 4096, "fp16", False, "shared 32x64"),   # 6.3 / 6.4 shared 64x64
    (256, 2048, 4096, "fp16", False, "shared 32x64"),   # 8.1 / 8.2 shared 64x64
    (256, 4096, 4096, "fp16", False, "shared 64x64"),   # 11.2 / 11.5 shared 32x64
    (64, 256, 4096, "fp32", False, "shared 32x32"),     # 9.1 / 9.5 small
    (128, 64, 4096, "fp32", False, "small"),            # 6.4 / 7.0 shared 32x64
    (256, 64, 4096, "fp32", False, "small"),            # 6.8 / 7.8 shared 32x64
    (256, 256, 4096, "fp32", False, "small"),           # 10.2 / 10.8 shared 32x64
    (256, 512, 4096, "fp32", False, "shared 32x64"),    # 11.6 / 13.0 small
    (256, 2048, 4096, "fp32", False, "shared 32x64"),   # 19.1 / 20.9 shared 64x64
    (128, 256, 4096, "fp16", True, "wide"),             # 5.3 / 5.5 shared 32x64
    (128, 512, 4096, "fp16", True, "shared 32x64"),     # 5.6 / 6.4 wide
    (256, 768, 2048, "fp16", True, "shared 32x64"),     # 6.4 / 7.5 wide
    (128, 1536, 4096, "fp16", True, "shared 32x64"),    # 7.8 / 7.8 shared 64x64
    (128, 2048, 4096, "fp16", True, "shared 64x64"),    # 8.1 / 8.4 shared 32x64
    (128, 4096, 4096, "fp16", True, "shared 64x64"),    # 10.9 / 11.7 shared 32x64
    (128, 768, 4096, "fp32", True, "shared 32x64"),     # 12.1 / 12.7 shared 64x64
])
def test_few_tiles_take_the_faster_one(M, K, N, dtype, two, tile):
    assert tile_of(M, K, N, dtype, two) == tile


@pytest.mark.parametrize("M,K,N,dtype,two,tile", [
    (512, 1536, 4096, "fp16", False, "wide"),           # 9.8 / 9.8 halves
    (640, 1792, 2048, "fp16", False, "wide"),           # 10.8 / 11.6 halves
    (640, 2048, 2048, "fp16", False, "halves"),         # 11.4 / 11.7 wide
    (640, 2816, 2048, "fp16", False, "wide"),           # 14.5 / 14.7 halves
    (640, 3072, 2048, "fp16", False, "halves"),         # 14.6 / 15.7 wide
    (640, 3328, 2048, "fp16", False, "halves"),         # 16.7 / 17.3 wide
    (512, 5504, 4096, "fp16", False, "halves"),         # 23.0 / 26.3 wide
    (1024, 1024, 5504, "fp16", False, "wide"),          # 13.3 / 15.7 flat
    (768, 512, 5504, "fp16", False, "wide"),            # 9.3 / 11.1 flat
    (768, 5504, 5504, "fp16", False, "wide"),           # 45.6 / 54.1 flat
    (2048, 512, 4096, "fp16", False, "wide"),           # 11.7 / 12.2 flat
    (1024, 256, 11008, "fp16", False, "flat"),          # 11.8 / 12.1 wide
    (1024, 2816, 4096, "fp16", False, "wide"),          # 20.6 / 20.5 groups
    (768, 2816, 4096, "fp16", False, "wide"),           # 19.0 / 19.7 groups
    (1024, 4096, 4096, "fp16", False, "groups"),        # 26.8 / 28.1 wide
    (1024, 1536, 4096, "fp32", False, "wide"),          # 38.0 / 38.7 groups
    (768, 2048, 4096, "fp32", False, "groups"),         # 43.3 / 43.9 wide
    (1024, 4096, 4096, "fp32", False, "groups"),        # 73.0 / 79.1 wide
    (512, 768, 2048, "fp16", True, "wide"),             # 7.7 / 8.3 halves
    (512, 1024, 2048, "fp16", True, "halves"),          # 8.2 / 8.8 wide
    (512, 2048, 2048, "fp16", True, "halves"),          # 11.3 / 13.1 wide
    (512, 768, 2048, "fp32", True, "wide"),             # 17.7 / 19.8 halves
    (512, 1024, 2048, "fp32", True, "halves"),          # 19.8 / 20.7 wide
    (512, 256, 4096, "fp16", True, "wide"),             # 6.9 / 7.2 flat
    (512, 1024, 4096, "fp16", True, "groups"),          # 11.1 / 11.7 flat
    (768, 2048, 2048, "fp16", True, "groups"),          # 15.5 / 17.2 flat
    (768, 1536, 4096, "fp16", True, "wide"),            # 20.0 / 20.3 flat
    (768, 5504, 4096, "fp16", True, "flat"),            # 57.2 / 59.4 wide
])
def test_more_tiles_take_the_faster_one(M, K, N, dtype, two, tile):
    assert tile_of(M, K, N, dtype, two) == tile


def test_planes_count_as_units_and_other_devices_have_their_own_lines():
    assert tile_of(128, 256, 4096, "fp16", planes=2) == tile_of(128, 512, 4096, "fp16") == "shared 32x64"
    assert tile_of(128, 256, 2048, "fp16", units=64) == tile_of(256, 256, 4096, "fp16")
    for bad in ((0, 8, 8, 1, 0, 0, 256), (64, 8, 8, 1, 2, 0, 256), (64, 8, 8, 0, 0, 0, 256), (64, 8, 8, 1, 0, 0, 0)):
        assert _lib.lib().tl_matrix_tile(*bad) < 0


# For each kind of call (rows, two weights) a size at which it takes each of its tiles, with rows, columns and a stage of K left over: what the
# GPU tests that have to reach every tile run (columns are even, K whole 16-byte pieces, for gated and chained calls).
SIZES = {
    ("fp16", False): {"shared 32x32": (97, 1408, 1002), "shared 32x64": (253, 1104, 3970), "shared 64x64": (250, 2312, 4002), "small": (130, 248, 4002),
                      "wide": (520, 1096, 2058), "halves": (450, 2040, 4002), "groups": (900, 3336, 4090), "flat": (2110, 264, 4090), "tall": (4093, 200, 4090)},
    ("fp32", False): {"shared 32x32": (97, 1408, 1002), "shared 32x64": (253, 1104, 3970), "small": (130, 248, 4002),
                      "wide": (520, 1096, 2058), "groups": (900, 2568, 4090), "flat": (2110, 264, 4090)},
    ("fp16", True): {"shared 32x32": (97, 1408, 1002), "shared 32x64": (200, 2056, 1034), "shared 64x64": (150, 2312, 2050), "wide": (520, 248, 2058),
                     "halves": (450, 1032, 2002), "groups": (500, 2616, 4090), "flat": (850, 2312, 4090), "tall": (4093, 200, 4090)},
    ("fp32", True): {"shared 32x32": (97, 1408, 1002), "shared 32x64": (200, 2056, 1034), "wide": (520, 248, 2058),
                     "halves": (450, 1032, 2002), "groups": (500, 2616, 4090), "flat": (1100, 264, 4090)},
}


@pytest.mark.parametrize("kind", list(SIZES))
def test_every_tile_has_a_size(kind):
    """A line that moves takes no tile out of the tests unnoticed; and no tile is reached that has none."""
    for tile, (M, K, N) in SIZES[kind].items():
        assert tile_of(M, K, N, *kind) == tile and N % 2 == 0 and K % 8 == 0
    reached = {tile_of(M, K, N, *kind) for M in (49, 97, 128, 250, 520, 900, 1100, 2110, 8192) for K in (8, 256, 512, 1024, 2048, 4096, 11008)
               for N in (8, 512, 1024, 2048, 4096, 11008)}
    assert reached == set(SIZES[kind])


def test_the_traffic_record_s_hash_covers_what_the_kernel_includes():
    import os
    import re

    import bench
    csrc = os.path.join(bench.ROOT, "ternaryllm_amd", "csrc")
    seen, todo = set(), ["tl_matrix.hip", "tl_layout.cpp"]
    while todo:
        name = todo.pop()
        if name in seen or not os.path.exists(os.path.join(csrc, name)):
            continue                                                 # (the interface's header is not of the kernel's own)
        seen.add(name)
        with open(os.path.join(csrc, name)) as f:
            todo += re.findall(r'#include "(.*?)"', f.read())
    assert seen == set(bench.KERNEL_SOURCES)
