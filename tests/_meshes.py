"""Meshes whose sweeps take each of the library's paths, with the strip plan
that each is expected to have: renumbered grids (rows of seven and eight lower
blocks, dependencies many sub-levels back), tubes and tori (rows with more
than 32 factor updates), grids whose sides sit at the edges of a strip."""
import numpy as np

from cloth_sim_self_collision_amd import scene


def grid(nx, ny):
    return scene.drop_on_obstacle(nx, 0.4, scene.sphere((0.0, 0.0, 0.0), 0.3), ny=ny, seed=nx + ny)


def renumbered(cl, order):
    """Vertex k of the result is vertex order[k] of cl."""
    order = np.asarray(order, np.int32)
    new = np.empty_like(order)
    new[order] = np.arange(cl.np_, dtype=np.int32)
    cl.xyz0 = cl.xyz0.reshape(-1, 3)[order].reshape(-1).copy()
    cl.xyz = cl.xyz.reshape(-1, 3)[order].reshape(-1).copy()
    cl.tri = new[cl.tri]
    cl.quad = scene.bending_quads(cl.tri)
    return cl


def shuffled(n):
    """A square grid with its vertices numbered at random."""
    return renumbered(grid(n, n), np.random.default_rng(n).permutation(n * n))


def jittered(nx, ny, window, seed):
    """A grid whose vertices changed places with others nearby in the order."""
    key = np.arange(nx * ny) + np.random.default_rng(seed).uniform(0, window, nx * ny)
    return renumbered(grid(nx, ny), np.argsort(key, kind="stable"))


def morton(n):
    """A square grid numbered along a Z-order curve."""
    x, y = np.repeat(np.arange(n), n), np.tile(np.arange(n), n)

    def spread(v):
        return sum(((v >> b) & 1) << (2 * b) for b in range(10))
    return renumbered(grid(n, n), np.argsort(spread(x) | spread(y) << 1, kind="stable"))


def tube(m, n, copies=1, closed=False):
    """Tubes of m vertices around and n along (closed: tori), side by side.
    Four around: rows with 35 factor updates; 3 x 3 tori, where every vertex
    couples to all others: 36.  A lane of the factorisation keeps updates 1 to
    32 of a row in registers.  (The tori pass through themselves, which the
    reference's impact zones never resolve: for assembly and solves only.)"""
    cl = grid(m, n * copies)
    a, c = np.meshgrid(np.arange(m), np.arange(n if closed else n - 1))
    p, q = c * m + a, c * m + (a + 1) % m
    r, s = (c + 1) % n * m + a, (c + 1) % n * m + (a + 1) % m
    tri = np.stack([p, q, s, p, s, r], -1).reshape(-1)
    cl.tri = np.concatenate([tri + k * m * n for k in range(copies)]).astype(np.int32)
    v = np.arange(m * n * copies)
    t, u, k = 2 * np.pi * (v % m) / m, v // m % n, v // (m * n)
    u = 2 * np.pi * u / n if closed else 0.02 * u
    xyz = [0.05 * np.cos(t) + (0.1 * np.cos(u) if closed else u) + 0.4 * k,
           0.05 * np.sin(t) + 0.3, 0.1 * np.sin(u) if closed else 0.05 * np.cos(t)]
    cl.xyz = np.stack(xyz, -1).reshape(-1)
    cl.xyz0 = cl.xyz.copy()
    cl.quad = scene.bending_quads(cl.tri)
    return cl


QUAD, ROWS = "quad", "rows"  # no strip plan: the packed one-workgroup sweep, the row-by-row sweep

# name: (mesh, expected (blocks per row, ring sub-levels, forward strips) or QUAD or ROWS)
MESHES = {
    "2x2": (lambda: grid(2, 2), (3, 8, 1)), "2x3": (lambda: grid(2, 3), (4, 8, 1)),
    "8x8": (lambda: grid(8, 8), (6, 8, 1)), "9x9": (lambda: grid(9, 9), (6, 8, 1)),
    "16x40": (lambda: grid(16, 40), (6, 8, 2)), "17x33": (lambda: grid(17, 33), (6, 8, 3)),
    "33x17": (lambda: grid(33, 17), (6, 8, 5)), "3x90": (lambda: grid(3, 90), (6, 8, 1)),
    "90x3": (lambda: grid(90, 3), (5, 8, 1)), "65x64": (lambda: grid(65, 64), (6, 8, 9)),
    "stack3x18": (lambda: scene.stacked_sheets(3, 18), (6, 8, 7)),
    "tube4x60": (lambda: tube(4, 60), (7, 16, 1)),
    "tori3x3": (lambda: tube(3, 3, 60, True), (8, 16, 8)),
    "morton64": (lambda: morton(64), (7, 16, 8)),
    "jitter24a": (lambda: jittered(24, 24, 1.5, 0), (7, 32, 4)),
    "jitter24b": (lambda: jittered(24, 24, 12, 0), (8, 16, 4)),
    "jitter24c": (lambda: jittered(24, 24, 4, 0), (8, 32, 4)),
    "jitter40": (lambda: jittered(40, 40, 12, 1), (8, 32, 25)),
    # a dependency lies further back than the ring
    "jitter40far": (lambda: jittered(40, 40, 1.5, 1), QUAD),
    "jitter40far8": (lambda: jittered(40, 40, 3, 0), QUAD),
    "shuffled20": (lambda: shuffled(20), ROWS),  # rows wider than eight lower blocks
}
