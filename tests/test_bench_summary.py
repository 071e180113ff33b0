"""What bench.py derives from counts: the operations of the sum-factorised
contraction."""
import bench


def test_operations_of_the_contraction():
    """F_SEP from the stages' definitions: nine jet slots in six x-y parts, six blocks,
    sixteen (qx, qy) pencils of four points."""
    parts, pencils, blocks = 6, 16, 6
    # z, per pencil and block: for every point, row slot, column part and cz the two-term
    # column sum (the second weight zero where a part has one slot), then bz
    z = 4 * 9 * parts * 3 * ((1 + 2) + 3 * 2)
    # y, per pencil and block: for every row part, (bz, cz) and cy the columns' sums over
    # dy' (three, two and one terms), then by
    y = parts * 9 * 3 * ((1 + 2 * 2) + (1 + 2) + 1 + 3 * 3 * 2)
    # x, per qx and block: for every (bz, cz), cy, by and cx the sums over dx' of three dx, then bx
    x = 9 * 3 * 3 * 3 * (3 * (1 + 2 * 2) + 3 * 3 * 2)
    assert bench.F_SEP == pencils * blocks * (z + y) + 4 * blocks * x
