"""CPU replay of the row-wise tiles that turn their tile in the first exchange
(RowTileStages / RowHalvesTileStages, ferrum-gpu_amd/csrc/kernels/fft_tile.hpp):
thread tid loads the positions t0 + T m of row c0 (c0 = tid / T, t0 = tid % T),
scatters its stage-0 outputs to that row of a [row][position] LDS tile and
gathers the positions t + T m of row c (c = tid % G, t = tid / G)."""

import pytest


def lds_pos(p):
    return p + (p >> 4)


def pitch(positions, g):
    return positions + positions // 16 + (1 if g >= 32 else 32 // g)


# (log2 length, rows per tile, elements per thread): 16 elements exchange the
# whole tile at once, 32 elements in two rounds of half the positions
TILES = [(7, 16, 16), (7, 64, 16), (9, 16, 32), (10, 16, 32)]


@pytest.mark.parametrize("log_l,g,e", TILES)
def test_first_exchange_turns_the_tile(log_l, g, e):
    n, rounds = 1 << log_l, e // 16
    t_n = n // e
    held = n // rounds
    p_row = pitch(held, g)
    threads = g * t_n
    assert p_row * g * 8 <= 160 * 1024
    got = {}
    for h in range(rounds):
        slots = {}
        for tid in range(threads):
            c0, t0 = divmod(tid, t_n)
            b = t0 + t_n * h                      # the thread's butterfly of this round
            assert (b < n // 16)
            for q in range(16):                   # output q at position 16 b + q
                pos = 16 * b + q
                assert held * h <= pos < held * (h + 1)
                slot = c0 * p_row + 17 * (b - held // 16 * h) + q
                assert slot == c0 * p_row + lds_pos(pos - held * h)
                assert 0 <= slot < p_row * g and slot not in slots
                slots[slot] = (c0, pos)
        assert len(slots) == g * held
        for tid in range(threads):
            c, t = tid % g, tid // g
            for m in range(16):
                d = t_n * m
                slot = c * p_row + lds_pos(t) + d + d // 16
                row, pos = slots[slot]
                assert (row, pos) == (c, t + t_n * (16 * h + m))
                got[(tid, 16 * h + m)] = pos
    assert len(got) == threads * e


@pytest.mark.parametrize("log_l,g,e", TILES)
def test_row_loads_cover_the_tile_in_contiguous_pieces(log_l, g, e):
    n = 1 << log_l
    t_n = n // e
    seen = set()
    for tid in range(g * t_n):
        c0, t0 = divmod(tid, t_n)
        for m in range(e):
            seen.add((c0, t0 + t_n * m))
    assert len(seen) == g * n
