"""The pieces in which the GPU tests prefill a prompt reach every way in which the attention's units are
merged (the plan is the library's own, qwen_layout.h, which layout_check covers exhaustively)."""

import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHECK = os.path.join(REPO, "qwen0.6b_amd", "layout_check")

# lengths of the calls that prefill one prompt, piece after piece
PIECES = [(15, 385, 200, 40, 260, 17, 183, 100, 200, 61, 239, 17, 323, 7),
          (450, 260, 190, 130, 70, 12, 100, 8, 140, 128, 62, 3, 147, 100, 240, 7)]


def test_pieces_reach_every_part_count():
    """Group units: items of 1 to 8 parts (5 to 8 reach into the second 1024-key chunk), two chunks in each
    of the builds for at most 16, 64, 128 and 256 positions. Chunk units: one and two."""
    if not os.path.exists(CHECK):
        pytest.skip("layout checker not built")
    groups, chunks, over = set(), set(), set()
    for sizes in PIECES:
        start = 0
        for n in sizes:
            out = subprocess.run([CHECK, "plan", str(n), str(start)], capture_output=True, text=True, check=True).stdout
            blocks, *parts = map(int, out.split())
            assert blocks in (4, 16)
            (groups if blocks == 4 else chunks).update(parts)
            if blocks == 4 and max(parts) > 4:
                over.add(next(c for c in (16, 64, 128, 256, 512, 1024) if n <= c))
            start += n
        assert 1024 < start <= 2047
    assert groups == set(range(1, 9))
    assert chunks == {1, 2}
    assert over >= {16, 64, 128, 256}
