"""Collision with 16 lanes per env (many envs of a small model), 64 lanes, and one lane per env (the single fused kernel's
variant 0, and very many envs of a small model) give the same bits, also where the broadphase buffer overflows."""
import numpy as np
import pytest
import torch

from genesis_amd import workloads as W
from genesis_amd.model import CompileOptions, compile_model
from tests.test_gpu_bodies import stacks

pytestmark = pytest.mark.gpu

COMPARED = ["qpos", "vel", "n_con", "n_contacts", "n_broad", "broad_pairs", "contact_geoms", "contact_pos", "contact_normal",
            "contact_pen", "cache_normal", "sort_value", "sort_ig", "aabb_min", "aabb_max", "errno_env"]
B = 2051  # 513 wavefronts of four envs, the last one partly filled


@pytest.mark.parametrize("name,pairs", [("quadruped", 300), ("arm", 300), ("boxes", 300), ("boxes", 1)])
def test_collision_lanes_agree(name, pairs):
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.rigid_solver import RigidSolver
    if name == "boxes":
        ents, q = stacks(7, 41, 5)
    else:
        ents = [W.plane_entity(), W.go2_entity() if name == "quadruped" else W.panda_entity()]
    M = compile_model(ents, CompileOptions(dt=0.005, max_collision_pairs=pairs))
    if name != "boxes":
        rng = np.random.default_rng(2)
        q = np.tile(np.asarray(M.qpos0, np.float64), (41, 1))
        if name == "quadruped":
            q[:, 2] = rng.uniform(0.05, 0.4, 41)  # from lying to hanging in the air
            q[:, 7:] += rng.uniform(-0.3, 0.3, (41, M.n_qs - 7))
        else:
            q[:, 1] = rng.uniform(1.2, 1.7, 41)  # the hand reaches the ground or stays clear of it
            q[:, 3] = rng.uniform(-0.3, -0.1, 41)
    q = torch.as_tensor(np.tile(q, (B // 41 + 1, 1))[:B], dtype=torch.float32)
    many, few, lane = (RigidSolver(M, n, "cuda", solver_variant=1, collide_variant=v, dyn_variant=1)
                       for n, v in ((B, 1), (41, 1), (41, 0)))
    for S in (many, few, lane):
        S.set_qpos(q[:S._B])
    fb = FusedBatch([Group(lane, envs_per_tile=1, solver_variant=1, collide_variant=0)])
    seen = 0
    for _ in range(3):
        many.substep()
        few.substep()
        fb.step()
        torch.cuda.synchronize()
        seen = max(seen, int(few.st.t["n_contacts"][0].max()))
        for k in COMPARED:
            a, b, c = (S.st.t[k] for S in (many, few, lane))
            if k in ("broad_pairs", "contact_geoms", "contact_pos", "contact_normal", "contact_pen"):
                # entries beyond an env's count are left over from earlier steps
                n = few.st.t["n_broad" if k == "broad_pairs" else "n_contacts"][0].long()
                per = {"broad_pairs": 1, "contact_geoms": 2, "contact_pos": 3, "contact_normal": 3, "contact_pen": 1}[k]
                keep = torch.arange(b.shape[0], device=b.device)[:, None] < per * n[None]
                a, b, c = (torch.where(keep, x[:, :41], torch.zeros_like(x[:, :41])) for x in (a, b, c))
            assert torch.equal(b, c), f"{k}: 64 lanes and one lane differ"
            assert torch.equal(a[..., :41], b), f"{k}: 16 and 64 lanes differ"
            if a.shape[-1] == B:
                assert torch.equal(a[..., 41:82], a[..., :41]) and torch.equal(a[..., -1], a[..., (B - 1) % 41]), k
    assert seen > 0
    assert bool((few.st.t["errno_env"] & 1).any()) == (pairs == 1)


@pytest.mark.parametrize("deep", [0.0, 0.02])
def test_many_pairs_agree(deep):
    """More convex pairs than lanes, carried over between chunks; deep ones are left to GJK/EPA among the others."""
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.rigid_solver import RigidSolver
    ents, q = stacks(70, 3, 9)
    M = compile_model(ents, CompileOptions(dt=0.005, max_collision_pairs=400))
    q = q.reshape(3, 70, 7)
    q[:, 3::8, 2] -= deep  # top boxes of every second column
    q = torch.as_tensor(q.reshape(3, -1), dtype=torch.float32)
    wave, lane = (RigidSolver(M, 3, "cuda", solver_variant=1, collide_variant=v, dyn_variant=1) for v in (1, 0))
    for S in (wave, lane):
        S.set_qpos(q)
    fb = FusedBatch([Group(lane, envs_per_tile=1, solver_variant=1, collide_variant=0)])
    wave.substep()
    fb.step()
    torch.cuda.synchronize()
    for k in COMPARED:
        a, b = wave.st.t[k], lane.st.t[k]
        if k in ("broad_pairs", "contact_geoms", "contact_pos", "contact_normal", "contact_pen"):
            n = wave.st.t["n_broad" if k == "broad_pairs" else "n_contacts"][0].long()
            per = {"broad_pairs": 1, "contact_geoms": 2, "contact_pos": 3, "contact_normal": 3, "contact_pen": 1}[k]
            keep = torch.arange(b.shape[0], device=b.device)[:, None] < per * n[None]
            a, b = (torch.where(keep, x, torch.zeros_like(x)) for x in (a, b))
        assert torch.equal(a, b), k
    pairs = wave.st.t["broad_pairs"][:int(wave.st.t["n_broad"][0, 0]), 0]
    assert int(((pairs >> 16) > 0).sum()) > 64  # geom 0 is the plane
    # without a cached normal the first step of either heap leaves some pairs to GJK/EPA
    assert bool((wave.st.t["errno_env"] & 0x100).any())


@pytest.mark.parametrize("n,B", [(1, 16384), (5, 32768)])
def test_lane_per_env_over_very_many_envs(n, B):
    """At the line where variant 0 goes over to a lane per env (2 and 6 geoms), the plain and the phased step give the bits of
    16 lanes; one env fewer still takes those."""
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.rigid_solver import RigidSolver
    ents, q = stacks(n, 41, 5)
    M = compile_model(ents, CompileOptions(dt=0.005, max_collision_pairs=20))
    q = torch.as_tensor(np.tile(q, (B // 41 + 1, 1))[:B], dtype=torch.float32)
    lane, many, phased = (RigidSolver(M, B, "cuda", solver_variant=1, collide_variant=v, dyn_variant=1) for v in (0, 1, 0))
    fewer = RigidSolver(M, B - 1, "cuda", solver_variant=1, collide_variant=0, dyn_variant=1)
    assert [S.kernel_name(1) for S in (lane, many, fewer)] == ["k_collide", "k_collide_wave<16>", "k_collide_wave<16>"]
    for S in (lane, many, phased):
        S.set_qpos(q)
    # two groups: whole tiles of 64 lanes, then one of three envs, which its wavefront takes as the 16-lane form does
    fb = FusedBatch([Group(phased, 0, B - 67, 1, 1, 0), Group(phased, B - 67, 67, 1, 1, 0)], phased=True)
    for _ in range(2):
        lane.substep()
        many.substep()
        fb.step()
    torch.cuda.synchronize()
    assert int(many.st.t["n_contacts"].min()) >= 4
    for k in COMPARED:
        a, b, c = (S.st.t[k] for S in (lane, many, phased))
        if k in ("broad_pairs", "contact_geoms", "contact_pos", "contact_normal", "contact_pen"):
            cnt = many.st.t["n_broad" if k == "broad_pairs" else "n_contacts"][0].long()
            per = {"broad_pairs": 1, "contact_geoms": 2, "contact_pos": 3, "contact_normal": 3, "contact_pen": 1}[k]
            keep = torch.arange(b.shape[0], device=b.device)[:, None] < per * cnt[None]
            a, b, c = (torch.where(keep, x, torch.zeros_like(x)) for x in (a, b, c))
        assert torch.equal(a, b), f"{k}: one and 16 lanes differ"
        assert torch.equal(c, b), f"{k}: phased and plain differ"
