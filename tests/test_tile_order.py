"""The order in which a workgroup goes through the tiles of its window: a model of the rule in plain Python against its two
promises -- every tile once, and one multiple of the period in every full window, so that overlapping windows agree in time."""
import pytest


def tiles_of_window(T, C, R, rows, tile):
    chunks = 1 if C % rows == 0 else rows // C if rows % C == 0 else (rows + C - 2) // C + 1
    span = (chunks + R) * C
    if span >= T:
        return 0
    aligned = C % tile == 0 or (rows % C == 0 and C * R % tile == 0)
    return (span + tile - 1 + (0 if aligned else tile - 1)) // tile


@pytest.mark.parametrize("rows,tile", [(128, 64), (64, 32), (128, 32)])
def test_every_tile_once_and_in_step(rows, tile):
    for C in (1, 7, 8, 10, 16, 24, 32, 50, 64, 96, 100, 128, 192, 256, 300):
        for R in (0, 1, 2, 5, 9):
            T = 5 * (C * (R + 2) + rows)
            P = tiles_of_window(T, C, R, rows, tile)
            assert P > 0 and tiles_of_window(C * (R + 1), C, R, rows, tile) == 0
            for q0 in range(0, T, rows):
                last = min(q0 + rows, T) - 1
                t0 = max(q0 // C - R, 0) * C // tile
                t1 = -(-min((last // C + 1) * C, T) // tile)
                f = -(-t0 // P) * P
                first = f if f < t1 else t0
                order, t = [], first
                for _ in range(t1 - t0):
                    order.append(t)
                    t = t0 if t + 1 == t1 else t + 1
                assert t == first and sorted(order) == list(range(t0, t1))
                assert t1 - t0 <= P                   # a window holds no residue twice
                if t1 - t0 == P:
                    assert first % P == 0
