"""Box grids of hexes, for tests that need a given number of dofs."""
import numpy as np

from femocs_amd import mesh as M


def box_grid(nx, ny, nz, jitter=0.0):
    """Nodes and (nx - 1)(ny - 1)(nz - 1) hexes (UCD order) of a box grid, inner nodes moved by up
    to `jitter` of a cell."""
    X = np.stack(np.meshgrid(*[np.linspace(0.0, n, n) for n in (nx, ny, nz)], indexing="ij"), -1).reshape(-1, 3)
    if jitter:
        inner = np.all((X > 0) & (X < [nx, ny, nz]), axis=1)
        X[inner] += np.random.default_rng(3).uniform(-jitter, jitter, (inner.sum(), 3))
    at = np.arange(nx * ny * nz).reshape(nx, ny, nz)
    lex = np.stack([at[a:nx - 1 + a, b:ny - 1 + b, c:nz - 1 + c].reshape(-1) for c in (0, 1) for b in (0, 1)
                    for a in (0, 1)], 1)
    ucd = np.empty_like(lex)
    ucd[:, M.UCD_TO_LEX] = lex
    return X, ucd.astype(np.int32)
