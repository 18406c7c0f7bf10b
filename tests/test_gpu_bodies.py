"""The free-body Newton solver at the sizes where it changes form: one body, two wavefronts per env up to 128 dofs and
four above, one body a lane up to 64 and two beyond; rows that store few of their bodies' entries (frictionloss)."""
import numpy as np
import pytest
import torch

from genesis_amd import workloads as W
from genesis_amd.model import CompileOptions, compile_model
from tests.sync import gpu_to_oracle

pytestmark = pytest.mark.gpu

TOL = 1e-4


def stacks(n, B, seed):
    """n boxes in columns of up to four, each 0.3 mm inside what it stands on, slightly turned; the columns touch in
    pairs, so the contact graph has cycles."""
    ents = W.pile_entities(n, np.random.default_rng(1))
    sizes = np.array([e.links[0].geoms[0].data[:3] for e in ents[1:]])
    rng = np.random.default_rng(seed)
    q = np.zeros((B, n, 7))
    for b in range(B):
        for i in range(n):
            col, level = divmod(i, 4)
            below = sizes[4 * col:i, 2].sum() - 3e-4 * (level + 1)
            x = 0.6 * (col // 2) + (0.5 * (sizes[i, 0] + sizes[i - 4, 0]) - 3e-4 if col % 2 else 0.0)
            yaw = rng.uniform(-0.01, 0.01)
            q[b, i] = [x + rng.uniform(-1e-4, 1e-4), 0.0, below + 0.5 * sizes[i, 2], np.cos(yaw / 2), 0, 0, np.sin(yaw / 2)]
    return ents, q.reshape(B, 7 * n)


@pytest.mark.parametrize("n,friction", [(1, True), (2, False), (10, True), (21, False), (22, True), (64, False), (70, False)])
def test_free_body_solver(n, friction):
    """Every step starts the oracles from the HIP state; bound as in the other wavefront parity tests: 1e-4, or 4x the
    largest FP32-vs-FP64 spread of the oracle in that env. Then the fused launch, one wavefront per env, must give the
    plain step's bits."""
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.rigid_solver import RigidSolver
    from oracle.oracle import Oracle
    B = 3
    ents, q = stacks(n, B, n)
    M = compile_model(ents, CompileOptions(dt=0.005, max_collision_pairs=400))
    solvers = [RigidSolver(M, B, "cuda", solver_variant=1, collide_variant=1, dyn_variant=1) for _ in range(2)]
    for S in solvers:
        S.set_qpos(torch.as_tensor(q, dtype=torch.float32))
        S.set_dofs_velocity(0.2 * (torch.rand((B, M.n_dofs), generator=torch.Generator().manual_seed(n)) - 0.5))
        if friction:
            S.set_dofs_frictionloss(np.where(np.arange(M.n_dofs) % 5 == 1, 0.05, 0.0))
    S = solvers[0]
    O, O64 = Oracle(M, B, 32), Oracle(M, B, 64)
    fb = FusedBatch([Group(solvers[1], envs_per_tile=1, solver_variant=1, collide_variant=1)])
    rows = 0
    for step in range(4):
        torch.cuda.synchronize()
        gpu_to_oracle(S, O)
        gpu_to_oracle(S, O64)
        S.substep()
        fb.step()
        O.run(1)
        O64.run(1)
        torch.cuda.synchronize()
        rows = max(rows, int(S.st.t["n_con"][0].max()))
        for name in ("qpos", "vel"):
            got, o, o64 = S.st.t[name].T.cpu().numpy(), O.get(name), O64.get(name)
            for b in range(B):
                bound = np.maximum(TOL + TOL * np.abs(o[b]), 4 * np.abs(o[b] - o64[b]).max() + TOL)
                assert (np.abs(got[b] - o[b]) <= bound).all(), f"step {step} env {b} {name}"
            assert torch.equal(S.st.t[name], solvers[1].st.t[name]), f"step {step} {name}: fused and plain differ"
    assert rows >= 12 * n, rows


def test_budgets_beyond_the_body_solver():
    """A Hessian budget that leaves no room for the free-body solver's arrays goes to the entity-block solver, which gives
    the same bits: the largest budget of ten boxes, against the default one."""
    from genesis_amd.rigid_solver import RigidSolver
    n, B = 10, 3
    ents, q = stacks(n, B, n)
    M = compile_model(ents, CompileOptions(dt=0.005, max_collision_pairs=400))
    D, E = M.n_dofs, M.n_entities
    rest = 4 * 6 * D + 16 * E + 4 * 3 * D + 4 * (9 * E + 6) + 4 * (6 * E + 257) + 64
    a, b = (RigidSolver(M, B, "cuda", solver_variant=1, wave_h_floats=h) for h in (None, (160 * 1024 - rest) // 4))
    for S in (a, b):
        S.set_qpos(torch.as_tensor(q, dtype=torch.float32))
    for _ in range(5):
        a.substep()
        b.substep()
    torch.cuda.synchronize()
    assert int(a.st.t["n_con"][0].max()) > 0 and int(a.st.t["solver_iters"].max()) > 0
    for k in ("qpos", "vel", "efc_force", "n_con"):
        assert torch.equal(a.st.t[k], b.st.t[k]), k
