"""diffusion2d's wave strips at sizes that are no multiple of a strip or a chunk (the last strip
and chunk are moved back over their neighbours', which must neither store nor sum twice):
n = 64 + 1, one strip and one column more on either strip width, an odd and an even remainder,
a remainder of one pair."""
import pytest

from helpers import run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
@pytest.mark.parametrize("n", [66, 79, 127, 130, 143, 254, 255, 258, 1000, 1001, 1538, 2050, 3599])
def test_diffusion2d_ragged(mode, n):
    shapes = {k: n * n for k in ("u", "ub", "un", "unb", "ud", "und", "ubd", "unbd")}
    shapes.update({k: 1 for k in ("loss", "lossb", "lossd", "lossbd")})
    print(f"diffusion2d_{mode} n={n}", flush=True)
    run_parity("diffusion2d", mode, shapes, dict(n=n))


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
@pytest.mark.parametrize("n", [130, 386])
def test_diffusion2d_ragged_views(mode, n):
    shapes = {k: n * n for k in ("u", "ub", "un", "unb", "ud", "und", "ubd", "unbd")}
    shapes.update({k: 1 for k in ("loss", "lossb", "lossd", "lossbd")})
    print(f"diffusion2d_{mode} n={n} offset=1", flush=True)
    run_parity("diffusion2d", mode, shapes, dict(n=n), offset=1)
