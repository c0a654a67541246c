"""bench.py's roofline of the FP64 solve counts what its kernel moves (CPU): a
mesh of at most 131 072 velocity rows is solved with every row in its thread's
registers, so an inner iteration moves five vectors and no matrix; a larger one
streams the matrix."""
import bench

NV, NNZ, NP = 131070, 2343944, 65536   # 256 x 256 elements


def _bytes(inner, uzawa, sizes):
    res = dict(recs=[dict(inner=inner, uzawa=uzawa, solve_ms=100.0)], sizes=sizes)
    rl = bench.roofline(res, "k_uzawa_fp64")
    assert abs(rl["achieved"] - rl["bytes_per_launch"] / 0.1 / 1e9) <= 1e-12 * rl["achieved"]
    return rl["bytes_per_launch"]


def test_held_rows_move_no_matrix_an_iteration():
    sizes = [(NV, NNZ, NP)]
    assert _bytes(1001, 7, sizes) - _bytes(1000, 7, sizes) == 5 * NV * 8
    assert _bytes(0, 0, sizes) == NNZ * 12
    per_uzawa = 2 * 4 * NV * 12 + 7 * NV * 8 + 12 * NP * 8
    assert _bytes(0, 3, sizes) == NNZ * 12 + 3 * per_uzawa


def test_larger_meshes_stream_it():
    sizes = [(4 * NV, 4 * NNZ, 4 * NP)]
    assert _bytes(1001, 7, sizes) - _bytes(1000, 7, sizes) == 4 * (NNZ * 12 + 11 * NV * 8)
