"""Tests of programs built from the reference's own sources are skipped only
where those sources are absent; a program missing beside them is a failure."""
import pytest

import conftest


@pytest.mark.parametrize("present", [False, True])
def test_a_missing_program_is_skipped_only_without_its_sources(monkeypatch, tmp_path, present):
    apps = conftest._apps()
    monkeypatch.setattr(apps, "REFERENCE", str(tmp_path))
    monkeypatch.setattr(conftest, "_apps", lambda: apps)
    if present:
        (tmp_path / "apps").mkdir()
    with pytest.raises(AssertionError if present else pytest.skip.Exception):
        conftest.reference_program(tmp_path / "airfoil_ref")
    exe = tmp_path / "built"
    exe.touch()
    assert conftest.reference_program(exe) == exe
