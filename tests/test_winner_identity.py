"""Recorded selection winners belong to the kernels and selection rules they were timed with, not only to the profile."""
import shutil

from utils import helix_runtime

A, B = (2, 128, 128, 64, 64, 0, 64), (2, 64, 64, 64, 64, 0, 64)
PROFILE = {A: 1.0, B: 0.4}


def pick(verified):
    return helix_runtime.tuned_config("MI355X_FP16", ("gemm", 512, 512, 512), PROFILE, lambda: A, lambda: verified)


def fresh_process(monkeypatch):
    monkeypatch.setattr(helix_runtime, "_winners", {})
    monkeypatch.setattr(helix_runtime, "_code_fingerprint", {})


def test_winner_is_not_handed_out_after_a_change_of_the_kernels(tmp_path, monkeypatch):
    monkeypatch.setattr(helix_runtime, "root_path", str(tmp_path))
    monkeypatch.delenv("HELIX_SELECTION", raising=False)
    sources = tmp_path / "src_template"
    shutil.copytree(helix_runtime.SRC_ROOT, sources)
    monkeypatch.setattr(helix_runtime, "SRC_ROOT", str(sources))
    fresh_process(monkeypatch)
    assert pick(B) == B
    fresh_process(monkeypatch)
    assert pick(A) == B                                          # the recorded winner
    template = sources / "MI355X_FP16" / "gemm.hip"
    template.write_text(template.read_text() + "// changed\n")
    fresh_process(monkeypatch)
    assert pick(A) == A                                          # other kernels: timed again


def test_winner_is_not_handed_out_after_a_change_of_the_rules(tmp_path, monkeypatch):
    monkeypatch.setattr(helix_runtime, "root_path", str(tmp_path))
    monkeypatch.delenv("HELIX_SELECTION", raising=False)
    scripts = tmp_path / "scripts"
    shutil.copytree(helix_runtime._SCRIPTS_DIR, scripts)
    monkeypatch.setattr(helix_runtime, "_find_include_dir", lambda found=helix_runtime._find_include_dir(): found)
    monkeypatch.setattr(helix_runtime, "_SCRIPTS_DIR", str(scripts))
    fresh_process(monkeypatch)
    assert pick(B) == B
    rules = scripts / "MI355X_FP16" / "MI355X_FP16_gemm.py"
    rules.write_text(rules.read_text() + "VERIFY_TOP = 3\n")
    fresh_process(monkeypatch)
    assert pick(A) == A
