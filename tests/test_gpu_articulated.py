"""Articulated models at the sizes where the wavefront kernels change form: the single-entity Newton solver (one lane
per dof up to 64 dofs, rows staged 64 at a time) against the CPU oracle."""
import numpy as np
import pytest
import torch

from genesis_amd import workloads as W
from genesis_amd.model import (CompileOptions, EntitySpec, JOINT_FREE, JOINT_PRISMATIC, JOINT_REVOLUTE, JointSpec,
                               LinkSpec, compile_model)
from tests.sync import gpu_to_oracle

pytestmark = pytest.mark.gpu

TOL = 1e-4


def chain_entity(n, free_base=False):
    """Chains of up to 12 one-dof links on a fixed or a floating base, n links in all (every fifth prismatic), with
    frictionloss on every joint and limits of +-0.05 on each fourth."""
    rng = np.random.default_rng(n)
    base_joint = JointSpec("base", JOINT_FREE, kp=0.0, kv=0.0, init_qpos=np.array([0, 0, 1.0, 1, 0, 0, 0])) if free_base \
        else JointSpec("base", 0)
    links = [LinkSpec("base", -1, np.array([0, 0, 1.0]), np.array([1.0, 0, 0, 0]), [base_joint], [], np.zeros(3),
                      np.array([1.0, 0, 0, 0]), np.eye(3) * 0.05, 4.0)]
    for i in range(n):
        axis = np.eye(3)[i % 3]
        limit = np.array([[-0.05, 0.05]]) if i % 4 == 0 else np.array([[-np.inf, np.inf]])
        j = JointSpec(f"j{i}", JOINT_PRISMATIC if i % 5 == 4 else JOINT_REVOLUTE, axis=axis, limit=limit, damping=0.1,
                      armature=0.1, stiffness=0.2, frictionloss=0.05, kp=5.0, kv=0.5)
        parent = 0 if i % 12 == 0 else i
        links.append(LinkSpec(f"l{i}", parent, rng.uniform(-0.05, 0.05, 3), np.array([1.0, 0, 0, 0]), [j], [],
                              rng.uniform(-0.02, 0.02, 3), np.array([1.0, 0, 0, 0]), np.diag(rng.uniform(0.5, 1, 3) * 1e-2),
                              rng.uniform(0.3, 1.0)))
    return EntitySpec(links, name="chain")


def start(S, M, B, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.as_tensor(np.tile(M.qpos0, (B, 1)), dtype=torch.float32)
    first = 7 if M.n_qs > M.n_dofs else 0  # the floating base stays where it is
    q[:, first:] += 0.3 * (torch.rand((B, M.n_qs - first), generator=g) - 0.5)
    S.set_qpos(q)
    S.set_dofs_velocity(torch.rand((B, M.n_dofs), generator=g) - 0.5)
    S.control_dofs_position(0.2 * (torch.rand((B, M.n_dofs), generator=g) - 0.5))


@pytest.mark.parametrize("n,free_base", [(7, False), (17, True), (33, False), (64, False), (65, False)])
def test_single_entity_solver_matches_oracle(n, free_base):
    """64 dofs is the last size with a lane per dof; its frictionloss and limit rows exceed the 64 staged at once. Each step starts the oracles from the HIP state; bound as in the other wavefront parity tests: 1e-4, or 4x
    the largest FP32-vs-FP64 spread of the oracle in that env."""
    from genesis_amd.rigid_solver import RigidSolver
    from oracle.oracle import Oracle
    M = compile_model([chain_entity(n, free_base)], CompileOptions(dt=0.005, enable_collision=False))
    B = 6
    S = RigidSolver(M, B, "cuda", solver_variant=1, wave_h_floats=4096)
    start(S, M, B, n)
    O, O64 = Oracle(M, B, 32), Oracle(M, B, 64)
    most = 0
    for step in range(4):
        torch.cuda.synchronize()
        gpu_to_oracle(S, O)
        gpu_to_oracle(S, O64)
        S.substep()
        O.run(1)
        O64.run(1)
        torch.cuda.synchronize()
        most = max(most, int(S.st.t["n_con"][0].max()))
        for name in ("qpos", "vel"):
            got, o, o64 = S.st.t[name].T.cpu().numpy(), O.get(name), O64.get(name)
            for b in range(B):
                bound = np.maximum(TOL + TOL * np.abs(o[b]), 4 * np.abs(o[b] - o64[b]).max() + TOL)
                assert (np.abs(got[b] - o[b]) <= bound).all(), f"step {step} env {b} {name}"
    assert most > (64 if n == 64 else 0), most


COMPARED = ["qpos", "vel", "acc", "acc_smooth", "dofs_pos", "links_pos", "links_quat", "geoms_pos", "geoms_quat",
            "aabb_min", "aabb_max", "cdof_ang", "cdof_vel", "cdofd_ang", "cdofd_vel", "root_com", "cd_vel", "cd_ang",
            "cinr_inertial", "cinr_pos", "cinr_mass", "links_iquat", "mass_blk", "mass_L_blk", "mass_D_inv",
            "qf_applied", "qf_passive", "qf_bias", "qf_smooth", "force", "xanchor", "xaxis", "errno_env"]


def _entities(name):
    if name == "quadruped":
        return [W.plane_entity(), W.go2_entity()]
    if name == "arm_boxes":  # an articulated entity beside free bodies: several blocks of the mass matrix
        return [W.plane_entity(), W.panda_entity()] + [W.box_entity((0.1, 0.1, 0.1), (0.6 + 0.3 * i, 0.5, 0.3)) for i in range(2)]
    n, free = name
    return [chain_entity(n, free)]


@pytest.mark.parametrize("name", ["quadruped", "arm_boxes", (7, False), (16, False), (17, False), (33, False), (11, True)],
                         ids=str)
@pytest.mark.parametrize("B", [1, 5, 1027])  # 64 lanes per env up to 1,024 envs, 16 above (1,027: a partial wavefront)
def test_tree_dynamics_equal_the_lane_per_env_ones(name, B):
    """step_1, step_2 and the kinematics refresh of articulated models spread over lanes give the bits of the one-lane
    walk: 16 dofs fill one register of the 16-lane substitutions, 17 two, 33 take the loop over LDS."""
    from genesis_amd.rigid_solver import RigidSolver
    M = compile_model(_entities(name), CompileOptions(dt=0.005, enable_self_collision=False,
                                                      enable_collision=isinstance(name, str)))
    out = []
    for dyn in (0, 1):
        S = RigidSolver(M, B, "cuda", solver_variant=1, collide_variant=1, dyn_variant=dyn)
        start(S, M, B, 3)
        for _ in range(3):
            S.substep()
        torch.cuda.synchronize()
        out.append({k: S.st.t[k].clone() for k in COMPARED})
    for k in COMPARED:
        assert torch.equal(out[0][k], out[1][k]), k


def test_trees_one_after_the_other_equal_the_plain_step():
    """Four envs of a tree whose four copies do not fit the LDS of a workgroup (40 dofs) take their turns on a wavefront of
    the fused kernel, in the same LDS words; the plain step gives each a wavefront of its own."""
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.rigid_solver import RigidSolver
    M = compile_model([chain_entity(40)], CompileOptions(dt=0.005, enable_collision=False))
    B = 9
    plain, fused = (RigidSolver(M, B, "cuda", solver_variant=1, dyn_variant=1) for _ in range(2))
    for S in (plain, fused):
        start(S, M, B, 7)
    fb = FusedBatch([Group(fused, envs_per_tile=4)])
    for _ in range(3):
        plain.substep()
        fb.step()
    torch.cuda.synchronize()
    for k in COMPARED:
        assert torch.equal(plain.st.t[k], fused.st.t[k]), k
