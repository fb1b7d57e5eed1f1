"""Grids beyond the library's limits are refused at tt_create, before any device work (checked without a GPU)."""
import pytest

from topopt_in_petsc_transient_amd import capi


@pytest.mark.parametrize("nel,word", [((1, 4095, 4095), "cross-section"), ((1000, 500, 400), "byte offsets"),
                                      ((1000, 1000, 1000), "dofs")])
def test_refused_grids(nel, word):
    with pytest.raises(capi.TTError) as e:
        capi.Context(capi.default_params(nelx=nel[0], nely=nel[1], nelz=nel[2], nlvls=1))
    assert e.value.code == -1 and word in str(e.value)
