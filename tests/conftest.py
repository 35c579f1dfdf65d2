import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))

# Tile choice must not depend on what a previous process cached: tests pin the
# library's heuristic pick unless they exercise the tuner themselves.
os.environ.setdefault("TRIFAST_AUTOTUNE", "0")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


class _ForcedTiles:
    """Calls of the operator with tiles of the test's choice.  ``forced({kernel: tile})``: from
    here on the kernels named run those tiles, the others the library's default ones.  The native
    host path remembers a shape's tiles and then no longer asks for them, so it starts with an
    empty memory and keeps nothing while the fixture is in use.  Before the next choice, and at
    the end of the test, every forced tile must have been launched since it was chosen (a dq tile
    under a dk/dv tile that writes dq itself is not launched, and must not be asked for)."""

    def __init__(self, monkeypatch):
        from trifast_amd import _lib, tuner
        from trifast_amd import torch as tt

        self._lib, self._tt = _lib.load(), tt
        self._q, self._kv = _lib.KERNEL_BWD_Q, _lib.KERNEL_BWD_KV
        self.tiles, self._asked = {}, {}
        self.launched = set()  # every (kernel, tile) so far
        tt._native().forget_tiles()
        monkeypatch.setattr(tuner, "pick", self._pick)
        monkeypatch.setattr(tt, "_tiles_to_keep", lambda q, tiles: False)

    def _pick(self, kernel, n, h, d, dtype, launch, extra_cost=None):
        tile = self.tiles.get(kernel)
        if tile is None:
            tile = self._lib.trifast_default_tile(kernel, n, h, d, self._tt._DTYPE_CODE[dtype])
        self._asked[kernel] = tile
        return tile

    def __call__(self, tiles):
        self.check()
        self.tiles, self._asked = dict(tiles), {}

    def check(self):
        launched = dict(self._asked)
        if self._kv in launched and self._lib.trifast_bwd_kv_tile_writes_dq(launched[self._kv]):
            launched.pop(self._q, None)
        for kernel, tile in self.tiles.items():
            assert launched.get(kernel) == tile, f"kernel {kernel}: tile {tile} was forced, {launched.get(kernel)} was launched"
        self.launched |= set(launched.items())


@pytest.fixture
def forced_tiles(monkeypatch):
    forced = _ForcedTiles(monkeypatch)
    yield forced
    forced.check()
