"""Recurrences over runs in chunks, several tiles of value columns a workgroup (so many heads that the columns are taken together): columns that end inside a tile,
tiles without columns, more than one workgroup a head."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,dk,dv,taps,ng", [(768, 1, 128, 33, 2, 1), (768, 2, 64, 48, 2, 1), (512, 1, 40, 65, 2, 2), (512, 2, 16, 100, 2, 1), (1200, 1, 100, 31, 2, 1)])
def test_any_cutting(H, G, dk, dv, taps, ng):
    import test_gpu_lelatar as lelatar

    for dtype in lelatar.DTYPES:
        lelatar.test_the_recurrence_carries_state_and_inputs_through_any_cutting(dtype, "ssd", H, G, dk, dv, taps, ng)
