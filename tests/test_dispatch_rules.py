"""Where the lines between kernels lie: answers of the library's rules at both sides of each, without a GPU."""
import pytest

from imparo_amd.kernels import library


@pytest.mark.parametrize("streams,width,top,pays", [
    (1, 4096, 0, 1), (2, 4096, 0, 1), (3, 1024, 0, 1), (3, 1280, 0, 0), (4, 1024, 0, 1), (4, 1280, 0, 0), (4, 4096, 0, 0),
    (1, 2048, 1, 1), (1, 2304, 1, 0), (2, 2048, 8, 1), (2, 2304, 8, 0), (4, 1024, 8, 1), (3, 1280, 2, 0)])
def test_a_step_norm_without_a_router(streams, width, top, pays):
    assert library().imparo_stream_step_takes(8, streams, width, 0 if top else 1, top)
    assert library().imparo_stream_step_pays(streams, width, top) == pays
