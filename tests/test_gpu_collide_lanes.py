"""Collision with 16 lanes per env (many envs of a small model), 64 lanes, and one lane per env (the single fused kernel's
variant 0, and very many envs of a small model) give the same bits, also where the broadphase buffer overflows."""
import numpy as np
import pytest
import torch

from genesis_amd import workloads as W
from genesis_amd.model import CompileOptions, compile_model
from tests.test_gpu_bodies import stacks

pytestmark = pytest.mark.gpu

# fields compared whole; the first `count` entries of lists (entries beyond are left over from earlier steps), by their width
WHOLE = ["qpos", "vel", "n_con", "n_contacts", "n_broad", "cache_normal", "sort_value", "sort_ig", "first_time", "aabb_min",
         "aabb_max", "errno_env"]
LISTS = {"broad_pairs": ("n_broad", 1), "contact_geoms": ("n_contacts", 2), "contact_pos": ("n_contacts", 3),
         "contact_normal": ("n_contacts", 3), "contact_pen": ("n_contacts", 1), "contact_friction": ("n_contacts", 1)}
ROWS = ["jac_nnz", "efc_diag", "efc_aref", "efc_D"]


def collided(S, n=None, first=0):
    """What the collision stage of n envs of S wrote (solver variant 1: rows env-major), blank beyond each env's counts."""
    t, M, dev = S.st.t, S.model, S.device
    envs = slice(first, first + (S._B if n is None else n))
    out = {k: t[k][:, envs].clone() for k in WHOLE}
    for k, (count, width) in LISTS.items():
        x = t[k][:, envs]
        keep = torch.arange(len(x), device=dev)[:, None] < width * t[count][0, envs].long()[None]
        out[k] = torch.where(keep, x, torch.zeros_like(x))
    R, W = M.max_rows, M.row_width
    con = t["n_con"][:, envs].long()
    row = torch.arange(R, device=dev)[None]
    live = row < con[0][:, None]
    for k in ROWS:
        x = t[k].reshape(S._B, R)[envs]
        out[k] = torch.where(live, x, torch.zeros_like(x))
    fl = (row >= con[1][:, None]) & (row < (con[1] + con[2])[:, None])
    x = t["efc_fl"].reshape(S._B, R)[envs]
    out["efc_fl"] = torch.where(fl, x, torch.zeros_like(x))
    entry = torch.arange(W, device=dev)[None, None] < out["jac_nnz"].long()[:, :, None]
    for k in ("jac_val", "jac_idx"):
        x = t[k].reshape(S._B, R, W)[envs]
        out[k] = torch.where(entry, x, torch.zeros_like(x))
    return out


def assert_same(a, b, what):
    for k in a:
        assert torch.equal(a[k], b[k]), f"{what}: {k}"


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
        a, b = collided(many, 41), collided(few)
        assert_same(b, collided(lane), "64 lanes and one lane")
        assert_same(a, b, "16 and 64 lanes")
        assert_same(collided(many, 41, 41), a, "two runs of 41 envs")
        assert_same(collided(many, 1, B - 1), collided(many, 1, (B - 1) % 41), "the last env")
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
    assert_same(collided(wave), collided(lane), "64 lanes and one lane")
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
    b = collided(many)
    assert_same(collided(lane), b, "one and 16 lanes")
    assert_same(collided(phased), b, "phased and plain")


@pytest.mark.parametrize("G,variant,kernel", [(1022, 0, "k_collide_wave<64>"), (1024, 1, "k_collide_wave<64>"),
                                              (1023, 0, "k_collide")])
def test_about_a_thousand_geoms(G, variant, kernel):
    """The largest models of the wavefront collision (64 KB of LDS, a little more where variant 1 asks for it) and the first
    beyond: two boxes on a bed of spheres, against a lane per env in the single fused kernel; the phased launch too."""
    from genesis_amd.batch import FusedBatch, Group
    from genesis_amd.model import GEOM_SPHERE, JOINT_FIXED, EntitySpec, GeomSpec, JointSpec, LinkSpec
    from genesis_amd.rigid_solver import RigidSolver
    one = np.array([1.0, 0, 0, 0])
    bed = [GeomSpec(GEOM_SPHERE, pos=np.array([0.1 * (i % 32), 0.1 * (i // 32), 0.05]), data=(0.05,)) for i in range(G - 3)]
    ents = [W.plane_entity(), EntitySpec([LinkSpec("bed", -1, np.zeros(3), one, [JointSpec("fix", JOINT_FIXED)], bed)], name="bed"),
            W.box_entity((0.25, 0.25, 0.1), (0.55, 0.55, 0.1495)), W.box_entity((0.2, 0.2, 0.2), (2.32, 1.37, 0.1995))]
    M = compile_model(ents, CompileOptions(dt=0.005, max_collision_pairs=40))
    assert M.n_geoms == G
    B = 3
    plain, lane, phased = (RigidSolver(M, B, "cuda", solver_variant=1, collide_variant=v, dyn_variant=1) for v in (variant, 0, variant))
    assert plain.kernel_name(1) == kernel
    fb = FusedBatch([Group(lane, envs_per_tile=2)])
    fp = FusedBatch([Group(phased, envs_per_tile=2)], phased=True)
    for _ in range(3):
        plain.substep()
        fb.step()
        fp.step()
    torch.cuda.synchronize()
    assert int(plain.st.t["n_contacts"].min()) >= 8  # four spheres under each box
    assert_same(collided(plain), collided(lane), "plain and one lane")
    assert_same(collided(phased), collided(lane), "phased and one lane")
