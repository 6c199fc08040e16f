"""Which tiles and slices the projections back to the hidden size take inside their launch: by what each was measured to take."""
import pytest


@pytest.mark.parametrize("hidden,form,rows", [
    (2048, None, 5), (4096, None, 5), (4224, None, 5), (4240, (4, 3), 1), (4608, (4, 3), 1), (5120, (4, 3), 1), (5376, (4, 3), 1), (5440, (4, 3), 1), (5456, None, 5), (6144, None, 5),
    (6336, None, 5), (6352, (4, 2), 9), (6656, (4, 2), 9), (8192, (4, 2), 9), (8208, None, 5), (8464, (8, 3), 9), (10880, (8, 3), 9), (10896, None, 5), (12288, None, 5)])
def test_forms(hidden, form, rows):
    from promptcache_amd.model.llama_hip import ks_forms
    assert ks_forms(hidden) == (form, form or (2, 2), rows)
