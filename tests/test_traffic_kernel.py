"""bench.py gives the measured HBM bytes of a tile shape only if they were measured on the kernel that the shape runs."""
import json

import pytest

import bench as B

NNZB = 159256


def test_recorded_kernel_is_the_shapes_kernel():
    with open(B.TRAFFIC_FILE) as f:
        shapes = json.load(f)["shapes"]
    for shape in B.FP32_SHAPES:
        assert shapes[",".join(map(str, shape))]["kernel"] == B.fp32_kernel(shape), shape


@pytest.mark.parametrize("shape", [(1, 32, 0), (2, 32, 2), (0, 32, 2)])
def test_bytes_of_another_kernel_are_no_figure(tmp_path, monkeypatch, shape):
    with open(B.TRAFFIC_FILE) as f:
        t = json.load(f)
    assert B.traffic_of(shape, NNZB) > 0
    t["shapes"][",".join(map(str, shape))]["kernel"] = "k_plane<float, 1, false, 16>"   # no shape runs this one
    other = tmp_path / "traffic.json"
    other.write_text(json.dumps(t))
    monkeypatch.setattr(B, "TRAFFIC_FILE", str(other))
    assert B.traffic_of(shape, NNZB) is None
