"""What a missing build of the reference's per-site code means (CPU)."""
import unittest

import pytest


def test_a_missing_reference_build_is_an_error_where_its_sources_are(monkeypatch, tmp_path):
    import oracle
    lib = str(tmp_path / "libjw_ref.so")
    monkeypatch.setattr(oracle, "REF_SRC", __file__)
    with pytest.raises(RuntimeError, match="reference build missing"):
        oracle.Reference(lib)


def test_without_the_sources_it_is_a_skip(monkeypatch, tmp_path):
    import oracle
    monkeypatch.setattr(oracle, "REF_SRC", str(tmp_path / "su3_matrix.h"))
    with pytest.raises(unittest.SkipTest):
        oracle.Reference(str(tmp_path / "libjw_ref.so"))
