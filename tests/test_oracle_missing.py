"""A size class whose reference build is not there: a missing file to a program, a skip to a test."""
import unittest

import pytest

import oracle_lib
from crm_inputs import make_case


def test_missing_reference_build(monkeypatch, tmp_path):
    monkeypatch.setattr(oracle_lib, "REF_DIR", str(tmp_path))
    case = make_case(1, 32, 28, 4000.0, 20.0)
    for kind in (FileNotFoundError, unittest.SkipTest):
        with pytest.raises(kind, match="libcrmref_32x1x28"):
            oracle_lib.reference(case)
