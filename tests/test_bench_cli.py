"""bench.py's command-line contract that needs no GPU."""

import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2
    assert "one GPU" in r.stderr
    assert r.stdout.strip() == ""


def test_pcg_byte_model_matches_the_kernels():
    sys.path.insert(0, ROOT)
    import bench
    matrix, couplings = 8 + 3 * 4, 3 * 4  # FP64 diagonal, FP32 face weights
    # FP64: z, s twice, q and x r/w with the matrix; r r/w, q, inverse diagonal,
    # factor and z; z r/w, inverse diagonal, factor and r.
    b = bench.KERNEL_BYTES["fp64"]
    assert b["k_spmv_dot"] == 6 * 8 + matrix
    assert b["k_forward"] == (2 + 1 + 1 + 3 + 1) * 8 and b["k_backward"] == (2 + 1 + 3 + 1) * 8
    assert sum(b.values()) == 188
    # FP32 MIC(0): the same in FP32 but x, which the forward sweep updates.
    b = bench.KERNEL_BYTES["mixed_mic0"]
    assert b["k_spmv_dot"] == 4 * 4 + matrix
    assert b["k_forward"] == (2 + 1 + 1 + 3 + 1 + 1) * 4 + 2 * 8 and b["k_backward"] == (2 + 1 + 3 + 1) * 4
    assert sum(b.values()) == 116
    # Multigrid, finest level: smoothings, restriction and correction each read
    # r, the inverse diagonal, the couplings and their vectors.
    b = bench.KERNEL_BYTES["mixed"]
    level = 4 + 4 + couplings
    assert b["k_spmv_dot"] == 3 * 4 + 8 + matrix
    assert b["k_axpy_norm"] == 5 * 8 + 2 * 4 + level
    assert b["k_forward"] == level + 4 + 4 / 8
    assert b["k_update_s"] == level + 4 + 4 + 4 / 8
    assert b["k_backward"] == level + 4 + 4 + 8
    # Level by level an eighth of that, with plain smoothings.
    down, up = level + 4, level + 4 + 4
    assert bench.COARSE_LEVEL_BYTES["mixed"] == (down + b["k_forward"] + b["k_update_s"] + up) / 7
    # A true residual: x, b, the matrix and r; in FP32 a forward sweep follows.
    assert bench.RESIDUAL_BYTES == {"fp64": 0, "mixed": 3 * 8 + matrix, "mixed_mic0": 2 * 8 + matrix + 4 + 6 * 4}
    for table in (bench.COARSE_LEVEL_BYTES, bench.RESIDUAL_BYTES, bench.KERNEL_NAMES):
        assert set(table) == set(bench.KERNEL_BYTES)
    # The paths change where the library's do.
    with open(os.path.join(ROOT, "flipengine3d_amd", "csrc", "scene.cpp")) as f:
        assert "constexpr size_t kMultigridCells = (size_t)1 << 20;" in f.read()
    assert bench.MULTIGRID_CELLS == 1 << 20
    args = bench.parse_args([])
    assert args.gpus == 1 and args.size == [256, 128, 128]
    assert json.dumps({"x": None})  # the line is plain JSON


def test_cpu_baseline_leaves_stdout_to_the_json_line():
    # The reference engine prints a banner and a log on stdout; bench.py's
    # stdout must carry only its one JSON line.
    code = ("import sys, json; sys.path.insert(0, %r); import bench; from flipengine3d_amd import scenes; "
            "a = bench.parse_args(['--size', '24', '16', '16', '--cpu-seconds', '0.01', '--cpu-threads', '1']); "
            "s = scenes.double_dam_break(24, 16, 16, 1 / 16, seed=3); r = bench.cpu_baseline(s, a); "
            "print(json.dumps(r))") % ROOT
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    lines = r.stdout.strip().splitlines()
    assert len(lines) == 1, r.stdout
    assert json.loads(lines[0])["value"] > 0
