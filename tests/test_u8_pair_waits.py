"""Requests and waits of the tiled u8 kernels that fetch two neighbouring chunks of weights and their one scale together
(see test_u8_waits.py, whose reader of the device code is used here)."""
import pytest

from test_u8_waits import device_code, slices  # noqa: F401 (a fixture)


# (rows, columns, wavefronts along them, groups)
TILES = [(256, 192, 4, 2, 1), (256, 128, 4, 2, 1), (128, 128, 4, 2, 1), (128, 64, 2, 2, 1), (64, 64, 2, 2, 1),
         (128, 64, 2, 2, 2), (64, 64, 2, 2, 4), (192, 192, 2, 4, 1), (192, 128, 2, 4, 1), (96, 96, 3, 2, 1)]


@pytest.mark.parametrize("tile", TILES, ids=lambda t: "%dx%d_%dx%d_k%d" % t)
def test_a_slice_waits_for_the_transfers_of_the_slice_before(device_code, tile):  # noqa: F811
    rows, columns, wm, wn, groups = tile
    transfers = rows * 8 // (wm * wn * 64)
    chunks = columns * 8 // (wm * wn * 64)
    weights = 2 * (chunks - chunks // 2)    # sixteen weights and their scale per pair of chunks, eight for an odd one
    prologue, loop = slices(device_code, f"gemm_nt_u8_pairs_kernelILi{rows}ELi{columns}ELi{wm}ELi{wn}ELb1ELi64ELi{groups}E")
    assert sorted(prologue[0]) == sorted("A" * 2 * transfers + "W" * 3 * weights)
    assert prologue[0].endswith("A" * transfers) and prologue[1] == transfers
    live, dead = "A" * transfers + "W" * weights, "A" * transfers
    assert [requests for requests, _ in loop].count(live) == 9, loop
    assert [requests for requests, _ in loop].count(dead) == 2 and len(loop) == 11, loop
    assert {count for _, count in loop} == {transfers + weights}
