"""The shapes of the bf16 GEMM's tile tests, against the table they are chosen by: the
launcher's cost rule is evaluated here on the table in its source, so that a change
of the table that leaves a tile without a test shows."""
import re

import numpy as np

from gpu_util import BF16_TILE_SHAPES
from metalbench_amd import helpers as H

SOURCE = (H.REPO_ROOT / "metalbench_amd" / "csrc" / "gemm_bf16.hip").read_text()


def _table():
    body = SOURCE[SOURCE.index("constexpr TileChoice k_tiles[]"):]
    rows = []
    for row in re.findall(r"\{TILE_([^}]*)\}", body[:body.index("};")]):
        kind, *v = [x.strip().rstrip("f") for x in row.split(",")]
        rows.append((kind, *[int(x) for x in v[:4]], *[np.float32(x) for x in v[4:]]))
    return rows


def _choose(m, n, k, odd):
    """The tile for A and B on (odd: off) and C on a 16-byte boundary."""
    best = None
    for kind, mb, nb, tm, tn, c0, c1, odd_c0, odd_c1, narrow in _table():
        slow = odd or k % 8 or n % 8 if kind == "REG" else odd
        if odd_c1 == 0 if slow else kind == "EDGE" and k % 8:
            continue
        tiles = -(-m // tm) * -(-n // tn)
        if tiles >= 1 << 23:
            continue
        base, step = (odd_c0, odd_c1) if slow else (c0, c1)
        more = narrow if n % (8 if kind == "EDGE" else 4) else np.float32(0)
        cost = np.float32((tiles + 255) // 256) * (base + step * np.float32(-(-k // 32)) + more)
        if best is None or cost < best[0]:
            best = (cost, (kind, mb, nb))
    return best[1]


def test_shapes_take_the_tiles_they_are_listed_for():
    for (m, n, k), even, odd in BF16_TILE_SHAPES:
        assert (even is None) == bool((n | k) & 1)
        if even:
            assert _choose(m, n, k, False) == even, (m, n, k)
        assert _choose(m, n, k, True) == odd, (m, n, k)


def test_every_tile_is_listed():
    table = _table()
    assert len(table) >= 10
    assert {e for _, e, _ in BF16_TILE_SHAPES if e} == {r[:3] for r in table}
    assert {o for _, _, o in BF16_TILE_SHAPES} == {r[:3] for r in table if r[8] != 0}
