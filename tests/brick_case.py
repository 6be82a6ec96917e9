"""The brick list's bricks of a system, counted on the host: own and staged atoms
of every brick of 4x4x4 list cells, as plan_grid, plan_bricks and k_brick_list
count them from the positions at the list's build."""
import numpy as np

R_INT = 3.72645          # outermost knot of the Fe potential
CELLS, CAP_MAX, THREADS = 216, 2560, (320, 384, 448, 512)


def threads_for(m):
    return next((t for t in THREADS if m <= t), 0)


def grid(sd, skin=0.3):
    """The list grid, rounded down to whole bricks where their atoms still fit."""
    b = sd.b0
    vol = abs(np.linalg.det(b))
    g = []
    for d in range(3):
        w = vol / np.linalg.norm(np.cross(b[:, (d + 1) % 3], b[:, (d + 2) % 3]))
        k = int(w / (R_INT + skin))
        g.append(min(k if k >= 3 else 1, 256))
    assert min(g) >= 4
    f = [k & ~3 for k in g]
    return f if threads_for(1.02 * 64.0 * sd.n / np.prod(f)) else g


def extents(sd, skin=0.3):
    """(own, staged) per brick; staged counts the 6x6x6 cells' atoms."""
    g = grid(sd, skin)
    c = np.minimum((sd.s - np.floor(sd.s)) * g, np.array(g) - 1).astype(int)
    cnt = np.zeros(g, int)
    np.add.at(cnt, tuple(c.T), 1)
    nb = [(k + 3) // 4 for k in g]
    own, staged = np.zeros(nb, int), np.zeros(nb, int)
    for b in np.ndindex(*nb):
        lo = [4 * k for k in b]
        own[b] = cnt[lo[0]:lo[0] + 4, lo[1]:lo[1] + 4, lo[2]:lo[2] + 4].sum()
        # cells -1..4 from the brick's first, up to one beyond the grid's end
        ix = [[x % g[d] for x in range(lo[d] - 1, min(lo[d] + 5, g[d] + 1))] for d in range(3)]
        staged[b] = cnt[np.ix_(*ix)].sum()
    return own.ravel(), staged.ravel()


def slab_with_gap(nc=(54, 54, 54), fill=0.6, seed=7):
    """A periodic box that a crystal fills along z, from just above the box's
    bottom (half a lattice spacing: no atom strays below) to the fraction fill."""
    from moldy_amd import lattice
    sd = lattice.make_system(nc=nc, sigma=0.08, temp=300.0, seed=seed)
    scale = np.array([1.0, 1.0, 1.0 / fill])
    s = sd.s + [0.0, 0.0, 0.5 / nc[2]]
    return lattice.System(b0=sd.b0 * scale, s=s / scale, x1=sd.x1 / scale, mass=sd.mass, z=sd.z,
                          deltat_fs=sd.deltat_fs)
