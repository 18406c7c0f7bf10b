"""Dynamics and kinematics of free bodies with (env, entity) lanes: workgroups of 1 to 4 envs by 64 entity lanes, of 4 by 32
and of 16 or more by 4, the last one partly filled, give the bits of the fused kernel's one-lane walk."""
import numpy as np
import pytest
import torch

from genesis_amd.model import CompileOptions, compile_model
from tests.test_gpu_articulated import COMPARED
from tests.test_gpu_bodies import stacks

pytestmark = pytest.mark.gpu


def same(a, b):
    if not a.is_floating_point():
        return torch.equal(a, b)
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("n,B", [(1, 3), (3, 1), (3, 5001), (20, 1030), (70, 5)])
def test_entity_lanes(n, B):
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.rigid_solver import RigidSolver
    ents, q = stacks(n, min(B, 7), n)
    M = compile_model(ents, CompileOptions(dt=0.005, max_collision_pairs=4 * n))
    q = torch.as_tensor(np.tile(q, (B // 7 + 1, 1))[:B], dtype=torch.float32)
    v = torch.rand((B, M.n_dofs), generator=torch.Generator().manual_seed(n)) - 0.5
    v[B // 2, -1] = float("nan")  # the last body's velocity: no body of that env moves
    plain, fused, fresh = (RigidSolver(M, B, "cuda", solver_variant=1, collide_variant=1, dyn_variant=d) for d in (1, 0, 1))
    for S in (plain, fused):
        S.set_qpos(q)
        S.set_dofs_velocity(v)
    fb = FusedBatch([Group(fused, envs_per_tile=1, solver_variant=1, collide_variant=1)])
    for _ in range(2):
        plain.substep()
        fb.step()
    torch.cuda.synchronize()
    for k in COMPARED:
        assert same(plain.st.t[k], fused.st.t[k]), k
    assert bool((plain.st.t["errno_env"].flatten() & 8).any())
    # the kinematics of a given pose
    fresh.set_qpos(plain.st.t["qpos"].T.contiguous())
    fresh.set_dofs_velocity(plain.st.t["vel"].T.contiguous())
    fresh.forward_kinematics()
    torch.cuda.synchronize()
    for k in ("links_pos", "links_quat", "geoms_pos", "geoms_quat", "root_com", "cinr_inertial", "cdof_ang", "cdof_vel",
              "cd_vel", "cd_ang"):
        assert same(fresh.st.t[k], plain.st.t[k]), k
