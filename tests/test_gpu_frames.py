"""Training frames whose lists outgrow their capacity: the frames are repeated with grown lists, and loss,
gradient and trained parameters are those of lists that fit from the start, bit for bit."""

import numpy as np
import pytest

from test_gpu_mlcg import cg_sim, hoomd  # noqa: F401
from test_gpu_mlp import cg_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cmax,nmax", [(2, 128), (64, 32), (2, 32)])
def test_overflow_repeats_the_frames(hoomd, cmax, nmax):  # noqa: F811
    from hoomd_amd import _lib
    N, out = 2500, []
    for shrink in (False, True):
        pos, L = cg_config(N, seed=4)
        sim, mlp, _ = cg_sim(hoomd, pos, L)
        sim.run(0)
        fs = hoomd.md.mlcg.FrameSet(2, N)
        rng = np.random.default_rng(9)
        for k in range(2):
            fs.set(k, cg_config(N, seed=20 + k)[0], rng.normal(0, 5, (N, 3)))
        if shrink:
            _lib.check(_lib.lib().hm_sys_set_list_capacity(sim._system, cmax, nmax))
        loss, grad = mlp.loss_grad(fs, 1)
        if shrink:
            _lib.check(_lib.lib().hm_sys_set_list_capacity(sim._system, cmax, nmax))
        losses = mlp.train(fs, 3, lr=1e-3, frames_per_step=2)
        sim.run(5)  # continues from the last frame
        out.append((np.array([loss]), grad, losses, mlp.params, mlp.forces))
    for a, b in zip(*out):
        assert np.array_equal(a, b) and np.isfinite(a).all()


@pytest.mark.parametrize("bad,code", [(np.nan, -4), (1e3, -5)])
def test_a_state_that_a_run_refuses_is_refused_by_training(hoomd, bad, code):  # noqa: F811
    from hoomd_amd import _lib
    N = 2500
    pos, L = cg_config(N, seed=4)
    sim, mlp, _ = cg_sim(hoomd, pos, L)
    sim.run(0)
    fs = hoomd.md.mlcg.FrameSet(1, N)
    fs.set(0, cg_config(N, seed=20)[0], np.zeros((N, 3)))
    loss, _ = mlp.loss_grad(fs, 0)
    wrong = np.array(pos)
    wrong[7, 1] = bad
    _lib.check(_lib.lib().hm_sys_set_state(sim._system, wrong.ctypes.data, None, None))
    for call in (lambda: mlp.loss_grad(fs, 0), lambda: mlp.train(fs, 1, lr=1e-3), lambda: sim.run(1)):
        with pytest.raises(_lib.HoomdAmdError) as e:
            call()
        assert e.value.code == code
    right = np.array(pos)
    _lib.check(_lib.lib().hm_sys_set_state(sim._system, right.ctypes.data, None, None))
    assert mlp.loss_grad(fs, 0)[0] == loss
