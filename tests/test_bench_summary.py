"""What bench.py derives from counts and counter files: the operations of the
sum-factorised contraction and the HBM summary of a counter run."""
import csv
import json

import pytest

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


def write_counters(path, counter, values):
    with open(path, "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value"])
        for i, (k, v) in enumerate(values):
            w.writerow([i, k, counter, v])


@pytest.mark.parametrize("tangent", ["void igap::k_tangent_sep<double, false>(igap::MeshK)",
                                     "void igap::k_tangent_gen<double, false>(igap::MeshK)"])
def test_counter_summary(tmp_path, monkeypatch, tangent):
    """The FP64 element tangent of a probe run, separable or general geometry, is found,
    and every assembly kernel's bytes are scaled by the calibration copy."""
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    (tmp_path / "profiles").mkdir()
    gather = "void igap::k_tangent_gather_rows<float, float>(igap::MeshK)"
    for name, scale in (("FETCH_SIZE", 1.0), ("WRITE_SIZE", 2.0)):
        write_counters(tmp_path / name, name, [("__amd_rocclr_copyBuffer", scale * bench.COPY_BYTES / 1024), (tangent, scale * 10.0),
                                               (tangent, scale * 30.0), (gather, scale * 7.0)])
    nel = (4, 3, 2)
    bench.pmc_json(nel, str(tmp_path / "FETCH_SIZE"), str(tmp_path / "WRITE_SIZE"))
    with open(tmp_path / "profiles" / "tangent_elem_4x3x2_pmc.json") as f:
        out = json.load(f)
    assert out["tangent_elem_bytes_per_launch"] == 2 * 20 * 1024
    assert bench.traffic_from_profiles(nel) == 2 * 20 * 1024
    assert bench.measured_bytes(nel, "igap::k_tangent_gather_rows<float, float>") == 2 * 7 * 1024
