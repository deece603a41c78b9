"""The host arithmetic of the network's transfers and launches (csrc/mlp_plan.h), in a program of its own
on the CPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "poe2d_amd", "csrc")


def run(tmp_path, body):
    src, exe = str(tmp_path / "t.cpp"), str(tmp_path / "t")
    with open(src, "w") as f:
        f.write('#include <cstdio>\n#include "mlp_plan.h"\nusing namespace poe2d::mlp;\nint main() {%s}\n' % body)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, src, "-o", exe], check=True)
    return [[int(v) for v in line.split()] for line in subprocess.run([exe], check=True, capture_output=True,
                                                                      text=True).stdout.splitlines()]


@pytest.mark.parametrize("floats,rows,cols", [(4096, 8, 5000), (4096, 8, 4096), (4096, 8, 4097), (4096, 5, 1000),
                                              (1, 3, 7), (524288, 64, 524289), (1 << 33, 200000, 20000)])
def test_a_staged_piece_fits_its_buffer_and_makes_progress(tmp_path, floats, rows, cols):
    # (a 5000 -> 8 network with batches of 32 has 4096 floats of workspace, less than one of its rows)
    (r, c), = run(tmp_path, f'auto p = staging_piece({floats}ull, {rows}, {cols}); printf("%d %d\\n", p.rows, p.cols);')
    assert 1 <= r <= rows and 1 <= c <= cols and r * c <= floats
    assert r == 1 or c == cols  # several rows only when whole: they are contiguous on the host
    assert c == cols or c == floats


@pytest.mark.parametrize("n,inputs,batch", [(37, 207, 1024), (2048, 207, 1024), (1 << 20, 256, 8192), (100000000, 207, 1024),
                                            (1000, 50000000, 32), (2147483647, 1, 32), (65536, 256, 8192), (65537, 256, 8192)])
def test_a_prediction_holds_bounded_inputs(tmp_path, n, inputs, batch):
    (rows,), = run(tmp_path, f'printf("%d\\n", predict_stretch({n}, {inputs}, {batch}));')
    assert 1 <= rows <= n
    assert rows * inputs <= max(1 << 24, batch * inputs)
    assert rows == n or (rows % batch == 0 and (rows + batch) * inputs > 1 << 24)


def test_output_layers_of_many_inputs_and_few_tiles_run_member_by_member(tmp_path):
    shapes = {(1024, 151500, 512): 1, (37, 6300, 512): 1, (1, 8, 4096): 1, (1, 8, 8192): 0, (64, 4032, 8192): 0,
              (65, 4032, 8192): 1, (64, 4096, 8192): 1, (256, 300, 65536): 0, (2147483647, 64, 1 << 24): 0}
    body = "".join(f'printf("%d\\n", ensemble_in_registers({m}, {n}, {k}));' for m, n, k in shapes)
    assert [v for v, in run(tmp_path, body)] == list(shapes.values())


def test_output_layers_of_one_member_run_split_from_2048_inputs_on(tmp_path):
    shapes = {(1, 8, 2048): 1, (1, 8, 2176): 0, (37, 300, 3072): 0, (256, 300, 3072): 1, (1, 8, 1 << 24): 0}
    body = "".join(f'printf("%d\\n", ensemble_in_registers({m}, {n}, {k}, true));' for m, n, k in shapes)
    assert [v for v, in run(tmp_path, body)] == list(shapes.values())
