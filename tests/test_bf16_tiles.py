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
    best = None
    for kind, mb, nb, tm, tn, c0, c1, odd_c0, odd_c1 in _table():
        if odd_c1 == 0 if odd else kind == "EDGE" and k % 8:
            continue
        tiles = -(-m // tm) * -(-n // tn)
        if tiles >= 1 << 23:
            continue
        base, step = (odd_c0, odd_c1) if odd else (c0, c1)
        cost = np.float32((tiles + 255) // 256) * (base + step * np.float32(-(-k // 32)))
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
    assert len(table) >= 9
    assert {e for _, e, _ in BF16_TILE_SHAPES if e} == {r[:3] for r in table}
    assert {o for _, _, o in BF16_TILE_SHAPES} == {r[:3] for r in table if r[8] != 0}
