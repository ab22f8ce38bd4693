"""The ray caster on the GPU (csrc/k_raycast.hip) where its launch and its stack
change: ray counts around a wave and around the blocks' turns on the XCDs, and
rays whose stack leaves LDS, against the oracle's traversal."""
import numpy as np
import pytest


def rays_through(rng, count, lo, hi):
    rays = np.zeros((count, 8), np.float32)
    a, b = rng.uniform(lo, hi, (2, count, 3))
    rays[:, 0:3], rays[:, 4:7] = a, b - a
    return rays


def deepest_stack(nodes, n, ray):
    """Entries on the path tracer's stack at most, with no triangle hit."""
    f = nodes.view(np.float32).reshape(n, 4, 4)
    ids = nodes.view(np.int32).reshape(n, 4, 4)[:, :, 3]
    o, d = ray[0:3], np.where(np.abs(ray[4:7]) < 1e-5, ray[4:7] + np.float32(1e-5), ray[4:7])
    stack, node, most = [], 0, 0
    while True:
        near = []
        if node >= 0:
            for s in (0, 1):
                t = np.sort((f[node, 2 * s:2 * s + 2, :3] - o) / d, axis=0)
                t0, t1 = t[0].max(), t[1].min()
                if t1 >= t0 and t1 >= 0:
                    near.append((t0, ids[node, 2 * s]))
            near.sort()
        stack += [c for _, c in near[1:]]
        most = max(most, len(stack))
        if not near and not stack:
            return most
        node = near[0][1] if near else stack.pop()


UNIT = np.array([0, 0, 0, 1, 1, 1], np.float32)  # the caller's bounds


def deep_mesh(rng):
    """Large overlapping triangles whose Morton keys are i ones and then zeros,
    i = 0 .. 30: a chain of a tree.  From beyond the upper corner the chain is
    always the nearer child, and every level leaves its other one behind."""
    keys = [((1 << i) - 1) << (30 - i) for i in range(31)]
    q = np.array([[sum((k >> (3 * b + axis) & 1) << b for b in range(10)) for axis in range(3)] for k in keys])
    c = (q + 0.5) / 1023.99
    e = rng.uniform(1.5, 2.0, (31, 3))
    tri = np.full((31, 3, 4), 3.1415, np.float32)
    tri[:, 0, :3], tri[:, 1, :3], tri[:, 2, :3] = c + e, c - e, c + e * [-0.9, 0.9, 0.3]
    return tri.reshape(31, 12)


def deep_rays(rng, count):
    return rays_through(rng, count, -1, 1) + np.float32([6, 6, 6, 0, -6, -6, -6, 0])


def test_deep_mesh_needs_more_than_the_lds_stack(ora):
    rng = np.random.default_rng(5)
    bvh = ora.build(deep_mesh(rng), UNIT, 0)[0]
    assert max(deepest_stack(bvh, 31, r) for r in deep_rays(rng, 200)) > 24


@pytest.mark.gpu
def test_rays_with_deep_stacks(ctx, ora):
    rng = np.random.default_rng(5)
    bvh, otri = ctx.build_arrays(deep_mesh(rng), UNIT)
    rays = deep_rays(rng, 3000)
    assert np.array_equal(ctx.raycast_arrays(bvh, otri, rays).view(np.uint32),
                          ora.raycast(bvh, otri, rays).view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 63, 64, 65, 32767, 32768, 32769, 70001])
def test_ray_counts(ctx, lb, ora, count):
    rng = np.random.default_rng(count)
    tri = lb.wl_clustered(count, 2000, 0.05)
    bvh, otri = ctx.build_arrays(tri, None)
    rays = rays_through(rng, count, 0.0, 1.0)
    assert np.array_equal(ctx.raycast_arrays(bvh, otri, rays).view(np.uint32),
                          ora.raycast(bvh, otri, rays).view(np.uint32))
