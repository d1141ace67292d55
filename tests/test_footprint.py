"""thy_footprint (no GPU): what a batch's HBM budget counts for a scenario."""
import pytest


# bytes a grid row of the tables: 8 + 16 + 24 values (row, face and deep-water records, the
# last padded to 32 bytes), 8 of the mass weight, 40 of Okada's
@pytest.mark.parametrize("precision,table", [(0, 32 + 64 + 96 + 48), (1, 64 + 128 + 192 + 48)])
@pytest.mark.parametrize("arrival", [False, True])
@pytest.mark.parametrize("nx", [56, 640, 4000])
def test_footprint_counts_every_row(nx, arrival, precision, table):
    from thysea import native
    pitch, esz = (nx + 63) // 64 * 64, 8 if precision else 4
    state = (9 if arrival else 8) * pitch * esz + nx * 12  # state block, Okada field, output field
    ny = 3000
    per_row = (native.footprint(nx, 2 * ny, precision, arrival) - native.footprint(nx, ny, precision, arrival)) / ny
    assert per_row >= state + table - 8
    lists = (nx + 55) // 56 * 8  # a work item for every three rows of a segment, twice over
    assert per_row <= state + table + 8 + lists
