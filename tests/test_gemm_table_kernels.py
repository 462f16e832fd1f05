"""Saved GEMM tables name the kernels that their variant numbers stand for (CPU): a table of other
kernels, such as the bare lists of earlier versions, is read but installs nothing."""
import json

import pytest

CHOICE = {"opA": "N", "opB": "C", "M": 792, "N": 792, "K": 1728, "batch": 1, "variant": 3, "split": 1,
          "seconds": 1e-4, "builtin_seconds": 2e-4}


@pytest.mark.parametrize("saved", [[CHOICE], {"kernels": ["64x64/16"], "choices": [CHOICE]}, {"choices": [CHOICE]}])
def test_tables_of_other_kernels(tmp_path, saved):
    from dirac_caspt2_amd import autotune
    from dirac_caspt2_amd.api import gemm_clear_choices
    path = tmp_path / "table.json"
    path.write_text(json.dumps(saved))
    gemm_clear_choices()
    with pytest.warns(UserWarning, match="other GEMM kernels"):
        assert autotune.load(str(path)) == 0
    assert gemm_clear_choices() == 0


def test_tables_of_these_kernels(tmp_path):
    from dirac_caspt2_amd import autotune
    from dirac_caspt2_amd.api import gemm_clear_choices
    path = tmp_path / "table.json"
    autotune.save([CHOICE], str(path))
    assert autotune.load(str(path)) == 1
    assert gemm_clear_choices() == 1
