"""The NCHW 1x1 kernel with rings of two, three and four stages: fewer steps than stages, as many, one
more, several rounds, and a last step of few channels; both sides of the line of two tiles a CU."""
import pytest

from test_gpu_conv_nchw import capi, run  # noqa: F401 (the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [None, 71, 72, 73, 74])
@pytest.mark.parametrize("channels", [64, 128, 144, 192, 448, 464, 512, 576, 848])
@pytest.mark.parametrize("n,h,w,o", [(1, 8, 12, 72), (2, 14, 14, 40), (3, 7, 7, 136)])
def test_rings(capi, cfg, channels, n, h, w, o):  # noqa: F811
    run(capi, (n, channels, h, w, o, 1, 1, 1, 0, 1), True, cfg=cfg)


@pytest.mark.parametrize("cfg", [72, 73, 74])
def test_rings_past_two_tiles_a_cu(capi, cfg):  # noqa: F811
    run(capi, (74, 528, 16, 16, 136, 1, 1, 1, 0, 1), False, cfg=cfg)
