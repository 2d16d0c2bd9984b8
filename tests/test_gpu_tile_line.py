"""The library's own tile choice on both sides of the latency layout's line for schemes of many registers."""
import pytest

from test_gpu_latency_layout import after, same

pytestmark = pytest.mark.gpu


# 1024 tiles of 8 x 8, the most that these schemes take the latency layout for, and 1056
@pytest.mark.parametrize("ni", [256, 257])
@pytest.mark.parametrize("flux,limiter,wavy", [("Roe", "superbee", False), ("M-AUSMPW+", "minmod", False),
                                               ("SLAU", "van_leer", False), ("SLAU", "van_leer", True)])
def test_library_choice_equals_an_explicit_tile(flux, limiter, wavy, ni):
    same(after(5, ni, 256, flux, limiter, wavy=wavy), after(5, ni, 256, flux, limiter, wavy=wavy, tile=2))
