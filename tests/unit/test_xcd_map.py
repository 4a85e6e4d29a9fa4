"""Bijection/coverage proof for the block maps of the attention kernels
(csrc/device.h): every (tile, head) pair is produced exactly once, and what
shares keys and values lands on one XCD.  xcd_tile_map serves prompts over
pages, latent prompts and training below 256 rows, head_tile_map training and
dense prompts, whose blocks are of unequal length; the latter is the source's
own, compiled for the CPU."""

import ctypes
import os
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(__file__), "..", "..", "csrc", "device.h")


def xcd_tile_map(block_id, nbx, grid):
    gy = grid // nbx
    if gy % 8 == 0:
        xcd, idx = block_id % 8, block_id // 8
        return idx % nbx, xcd + 8 * (idx // nbx)
    return block_id % nbx, block_id // nbx


@pytest.mark.parametrize("nbx,gy", [
    (16, 32),   # 1024 rows in tiles of 64, 32 heads
    (32, 64),
    (4, 192),   # 200 rows of 16 x 12 heads: two tiles; four
    (2, 4),     # gy % 8 != 0 -> identity
    (8, 96),
    (1, 8),
])
def test_xcd_map_bijective_and_affine(nbx, gy):
    grid = nbx * gy
    seen = set()
    bh_to_xcd = {}
    for bid in range(grid):
        bx, bh = xcd_tile_map(bid, nbx, grid)
        assert 0 <= bx < nbx and 0 <= bh < gy, (bid, bx, bh)
        assert (bx, bh) not in seen, "duplicate mapping"
        seen.add((bx, bh))
        if gy % 8 == 0:
            # affinity: all tile-blocks of one bh on one XCD (id % 8)
            xcd = bid % 8
            assert bh_to_xcd.setdefault(bh, xcd) == xcd, bh
    assert len(seen) == grid  # every (tile, bh) covered exactly once


@pytest.fixture(scope="module")
def head_tile_map(tmp_path_factory):
    text = open(HEADER).read()
    begin = text.index("DEVINL void head_tile_map")
    body = text[begin:text.index("\n}\n", begin) + 3]
    src = tmp_path_factory.mktemp("map") / "map.cpp"
    src.write_text("struct { unsigned x; } blockIdx;\n"
                   + body.replace("DEVINL", "static")
                   + """
extern "C" void blocks(int n, int nbx, int B, int H, int G, int* out) {
  for (int i = 0; i < n; ++i, out += 3) {
    blockIdx.x = i;
    head_tile_map(nbx, B, H, G, out, out + 1, out + 2);
  }
}
""")
    lib = str(src.with_suffix(".so"))
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", str(src), "-o", lib])
    return ctypes.CDLL(lib).blocks


@pytest.mark.parametrize("nbx,B,H,G", [
    (32, 2, 32, 8),    # 4096 rows, 8 pairs of kv heads: heads of a kv head together
    (32, 2, 8, 8),     # the same by kv heads (dK, dV)
    (8, 16, 12, 12),   # 1024 rows, 192 heads
    (3, 3, 12, 12),    # 36 heads: not a multiple of 8
    (4, 1, 5, 1), (2, 8, 7, 1), (6, 4, 6, 2), (5, 2, 24, 4), (1, 1, 1, 1), (1, 8, 40, 5),
])
def test_head_tile_map(head_tile_map, nbx, B, H, G):
    n = nbx * B * H
    flat = (ctypes.c_int * (3 * n))()
    head_tile_map(n, nbx, B, H, G, flat)
    got = [tuple(flat[3 * i:3 * i + 3]) for i in range(n)]
    # all heads' blocks of one tile, then all of the next
    assert [t for t, _, _ in got] == [i // (B * H) for i in range(n)]
    assert set(got) == {(t, b, h) for t in range(nbx) for b in range(B) for h in range(H)}
    if B * G % 8 == 0:
        xcd = {}
        for i, (_, b, h) in enumerate(got):
            assert xcd.setdefault((b, h // (H // G)), i % 8) == i % 8
