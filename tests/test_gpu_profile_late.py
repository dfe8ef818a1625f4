"""A launch of SOR sweeps whose waves wait longer than they may (here for no
longer than 64 polls, AX_SOR_SPINS) is given up, and the call goes on with one
wave a launch: the profile, the sweep count and the residual of an undisturbed
call."""
import numpy as np
import pytest

import axions_amd as ax
from oracle import oracle_py as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,tol,max_iter", [(301, 1e-12, 1500), (301, 1e-4, 4000), (40, 1e-9, 700), (130, 1e-6, 64)])
def test_waves_that_give_up(nx, tol, max_iter, monkeypatch):
    args = dict(nx=nx, h=0.05, w=1.5, tol=tol, n=1.0, lam=1.0, eta=1.0, g=0.7, max_iter=max_iter)
    want, wit, wres = orc.sor_profile(*(args[k] for k in ("nx", "h", "w", "tol", "n", "lam", "eta", "g", "max_iter")))
    for spins in (None, "0"):
        print(f"[sor late] nx={nx} max_iter={max_iter} spins={spins}", flush=True)
        if spins:
            monkeypatch.setenv("AX_SOR_SPINS", spins)
        prof, it, res = ax.sor_profile(**args)
        assert it == wit and res == wres
        assert np.array_equal(prof.view(np.uint64), want.view(np.uint64))
