"""bench.py divides counted HBM bytes by a measured step time: the count must be of the kernels that ran."""
import os
import shutil

import bench


def _profile(folder, sources):
    with open(os.path.join(folder, "hbm_traffic_w.md"), "w") as f:
        f.write('# counted\n\n```json\n{"step_sources": "%s", "total_GB_per_step": 1.0, "families": {}}\n```\n' % sources)


def test_a_count_of_other_kernels_is_not_used(tmp_path):
    assert bench.measured_traffic("w", str(tmp_path)) is None
    _profile(tmp_path, "0123456789abcdef")
    assert bench.measured_traffic("w", str(tmp_path)) is None
    _profile(tmp_path, bench.step_sources())
    assert bench.measured_traffic("w", str(tmp_path))["total_GB_per_step"] == 1.0


def test_the_fingerprint_follows_the_step_s_code_alone(tmp_path, monkeypatch):
    csrc = tmp_path / "css-code_amd" / "csrc"
    shutil.copytree(os.path.join(bench.ROOT, "css-code_amd", "csrc"), csrc, ignore=shutil.ignore_patterns("_build"))
    before = bench.step_sources()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.step_sources() == before
    for name, text, same in (("cssx_rhs.hip", "\n// a comment\n/* another\n one */\n", True), ("cssx_patches.hip", "\nint x;\n", True),
                             ("cssx_rhs_line.hpp", "\nint x;\n", False)):
        with open(csrc / name, "a") as f:
            f.write(text)
        assert (bench.step_sources() == before) == same, name


def test_the_final_kernel_by_its_rule():
    assert [bench.final_kernel(n, "f32", False) for n in (31, 32, 33)] == ["k_rhs_final", "k_rhs_line", "k_rhs_line"]
    assert [bench.final_kernel(n, "f64", False) for n in (47, 48, 50, 52)] == ["k_rhs_final", "k_rhs_line", "k_rhs_final", "k_rhs_line"]
    assert bench.final_kernel(512, "f32", True) == "k_rhs_final"
