"""Constraint impedance at the powers with a form of their own (0 to 4) and without (2.5, 5), in contact rows and in the
limit rows of an arm whose joints are spread over lanes."""
import numpy as np
import pytest
import torch

from genesis_amd import workloads as W
from genesis_amd.model import CompileOptions, compile_model
from tests.sync import gpu_to_oracle
from tests.test_gpu_bodies import stacks

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _steps(M, q, steps, need):
    """Steps from the HIP state; bound as in the other parity tests: 1e-4, or 4x the FP32-vs-FP64 spread of the oracle."""
    from genesis_amd.rigid_solver import RigidSolver
    from oracle.oracle import Oracle
    B = len(q)
    S, O, O64 = RigidSolver(M, B, "cuda", solver_variant=1, collide_variant=1), Oracle(M, B, 32), Oracle(M, B, 64)
    S.set_qpos(torch.as_tensor(q, dtype=torch.float32))
    for step in range(steps):
        torch.cuda.synchronize()
        gpu_to_oracle(S, O)
        gpu_to_oracle(S, O64)
        S.substep()
        O.run(1)
        O64.run(1)
        torch.cuda.synchronize()
        if step == 0:
            assert int(S.st.t["n_con"][0].min()) >= need
        for name in ("qpos", "vel"):
            got, o, o64 = S.st.t[name].T.cpu().numpy(), O.get(name), O64.get(name)
            for b in range(B):
                bound = np.maximum(TOL + TOL * np.abs(o[b]), 4 * np.abs(o[b] - o64[b]).max() + TOL)
                assert (np.abs(got[b] - o[b]) <= bound).all(), f"step {step} env {b} {name}"


@pytest.mark.parametrize("power", [1.0, 2.0, 2.5, 3.0, 4.0, 5.0])
def test_impedance_powers(power):
    ents, q = stacks(4, 3, 1)
    for e in ents:
        for l in e.links:
            for g in l.geoms:  # penetrations of 0.3 mm lie inside the width of 1 mm
                g.sol_params = np.array([0.02, 1.0, 0.5, 0.95, 0.001, 0.4, power])
    _steps(compile_model(ents, CompileOptions(dt=0.005)), q, 3, 16)
    arm = W.panda_entity()
    for l in arm.links:
        for j in l.joints:
            j.sol_params = np.array([0.02, 1.0, 0.5, 0.95, 0.05, 0.4, power])
    M = compile_model([arm], CompileOptions(dt=0.005, enable_collision=False))
    lim = np.asarray(M.dof_limit, np.float64)
    # every second joint up to 0.03 beyond its upper limit (fingers: 0.01)
    q = np.tile(lim.mean(1), (3, 1))
    over = np.array([0.03, 0.02, 0.01])[:, None] * np.where(np.arange(M.n_dofs) < 7, 1.0, 0.3)
    q[:, ::2] = (lim[:, 1] + over)[:, ::2]
    _steps(M, q, 3, (M.n_dofs + 1) // 2)
