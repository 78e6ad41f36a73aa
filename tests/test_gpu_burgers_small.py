"""burgers1d's one-wave blocks for small grids (csrc/burgers1d.hip) against the oracle: grids one
cell short of and past a block's 64, 128 or 192 cells, grids smaller than the 32-cell halo,
and both sides of the sizes at which each kernel's rule changes over (98304, 262144, 524288
cells), over a full 32-step chunk and a remainder."""
import pytest

from helpers import run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
@pytest.mark.parametrize("n", [3, 31, 63, 64, 65, 127, 129, 191, 193, 98304, 98305, 262145, 524289])
def test_burgers1d_small_grids(mode, n):
    T = 40 if n < 1000 else 34
    shapes = {k: n for k in ("u", "ub", "un", "unb", "ud", "ubd", "und", "unbd")}
    shapes.update({k: 1 for k in ("loss", "lossb", "lossd", "lossbd")})
    scalars = dict(nu=0.05, dt=0.002, dx=0.5, tend=10.0, nud=0.3, dtd=-0.2, dxd=0.1, tendd=0.7)
    stacks = () if mode == "d" else (("branch_stack", (T, "Ai")), ("u_stack", (T * n, "Af")))
    print(f"burgers1d_{mode} n={n} nsteps={T}", flush=True)
    run_parity("burgers1d", mode, shapes, dict(n=n, nsteps=T), scalars=scalars, stacks=stacks)
