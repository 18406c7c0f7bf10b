"""The free-body Newton solver at the sizes where it changes form: one body, two wavefronts per env up to 128 dofs and
four above, one body a lane up to 64 and two beyond; rows that store few of their bodies' entries (frictionloss, and the
partial chains of arms with six joints, whose six dofs are a body to this solver)."""
import numpy as np
import pytest
import torch

from genesis_amd import workloads as W
from genesis_amd.model import (EQ_CONNECT, EQ_JOINT, GEOM_CAPSULE, JOINT_FIXED, JOINT_REVOLUTE, CompileOptions, EntitySpec,
                               EqualitySpec, GeomSpec, JointSpec, LinkSpec, compile_model)
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


def six_joint_arm(name, x, y):
    """A chain of six capsules standing at (x, y); frictionloss on every other joint, limits of 0.03 on each third."""
    one = np.array([1.0, 0, 0, 0])
    links = [LinkSpec(f"{name}_base", -1, np.array([x, y, 0.1]), one, [JointSpec(f"{name}_fix", JOINT_FIXED)], [], np.zeros(3),
                      one, np.eye(3) * 0.05, 4.0)]
    for i in range(6):
        limit = np.array([[-0.03, 0.03]]) if i % 3 == 0 else np.array([[-np.inf, np.inf]])
        j = JointSpec(f"{name}_j{i}", JOINT_REVOLUTE, axis=np.array([[0.0, 1.0, 0.0], [1.0, 0.0, 0.0]][i % 2]), limit=limit,
                      damping=0.1, armature=0.1, kp=20.0, kv=2.0, frictionloss=0.05 * (i % 2))
        links.append(LinkSpec(f"{name}_l{i}", i, np.array([0, 0, 0.15 if i else 0.0]), one, [j],
                              [GeomSpec(GEOM_CAPSULE, pos=np.array([0, 0, 0.075]), data=(0.03, 0.1))], np.array([0, 0, 0.07]),
                              one, np.eye(3) * 1e-2, 1.0))
    return EntitySpec(links, name=name)


@pytest.mark.parametrize("scene", ["arms", "arm_boxes"])
def test_six_joint_arms(scene):
    """Rows that hold a part of a chain: two arms leaning on each other along their links (contacts of up to 6 + 6 entries),
    joined by a CONNECT, with a JOINT equality that names the later joint first; or one arm with boxes against its middle
    links; limit and frictionloss rows. Against the oracles as above, and bit by bit against the fused launch and the
    entity-block solver, which reads the rows as they are."""
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.rigid_solver import RigidSolver
    from oracle.oracle import Oracle
    B = 4
    a = six_joint_arm("a", 0.0, 0.0)
    if scene == "arms":
        b = six_joint_arm("b", 0.004, 0.0585)
        b.equalities = [EqualitySpec(EQ_JOINT, "b_j4", "b_j1", data=np.array([0.0, 1.0, 0, 0, 0])),
                        EqualitySpec(EQ_CONNECT, "b_l3", "a_l2", data=np.array([0.0, 0.0, 0.1]))]
        ents = [W.plane_entity(), a, b]
    else:
        # resting on nothing, moving towards the arm's side at the heights of its second and fourth link
        ents = [W.plane_entity(), a] + [W.box_entity((0.1, 0.08, 0.06), (0.01, s * 0.0695, z), rho=500.0)
                                        for s, z in ((1.0, 0.33), (-1.0, 0.62))]
    M = compile_model(ents, CompileOptions(dt=0.005))
    D, E = M.n_dofs, M.n_entities
    limit = (160 * 1024 - (4 * 6 * D + 16 * E + 4 * 3 * D + 4 * (9 * E + 6) + 4 * (6 * E + 257) + 64)) // 4
    solvers = [RigidSolver(M, B, "cuda", solver_variant=1, wave_h_floats=h) for h in (None, None, limit)]
    assert [S.kernel_name(2) for S in solvers] == ["k_solve_bodies<2>", "k_solve_bodies<2>", "k_solve_wave"]
    rng = np.random.default_rng(4)
    q = np.tile(M.qpos0.astype(np.float64), (B, 1))
    n_arm = 12 if scene == "arms" else 6
    q[:, :n_arm] += rng.uniform(-0.002, 0.002, (B, n_arm))
    q[:, 0] = 0.035  # beyond its limit
    v = rng.uniform(-0.1, 0.1, (B, D))
    if scene == "arm_boxes":
        v[:, 7], v[:, 13] = -0.3, 0.3
    for S in solvers:
        S.set_qpos(torch.as_tensor(q, dtype=torch.float32))
        S.set_dofs_velocity(torch.as_tensor(v, dtype=torch.float32))
    S = solvers[0]
    O, O64 = Oracle(M, B, 32), Oracle(M, B, 64)
    fb = FusedBatch([Group(solvers[1], envs_per_tile=1)])
    nnz = set()
    for step in range(6):
        torch.cuda.synchronize()
        gpu_to_oracle(S, O)
        gpu_to_oracle(S, O64)
        S.substep()
        fb.step()
        solvers[2].substep()
        O.run(1)
        O64.run(1)
        torch.cuda.synchronize()
        # the entity-block solver leaves the rows as the collision wrote them
        con = solvers[2].st.t["n_con"][0].cpu().numpy()
        for b, row in enumerate(solvers[2].st.t["jac_nnz"].reshape(B, M.max_rows).cpu().numpy()):
            nnz |= set(row[:con[b]].tolist())
        for name in ("qpos", "vel"):
            got, o, o64 = S.st.t[name].T.cpu().numpy(), O.get(name), O64.get(name)
            for b in range(B):
                bound = np.maximum(TOL + TOL * np.abs(o[b]), 4 * np.abs(o[b] - o64[b]).max() + TOL)
                assert (np.abs(got[b] - o[b]) <= bound).all(), f"step {step} env {b} {name}"
            for k, what in ((1, "fused"), (2, "entity blocks")):
                assert torch.equal(S.st.t[name], solvers[k].st.t[name]), f"step {step} {name}: {what}"
    print(f"{scene}: rows of {sorted(nnz)} entries")
    assert nnz & {7, 8, 9, 10, 11} and 1 in nnz and (scene != "arms" or 2 in nnz), nnz
