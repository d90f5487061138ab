"""Face samples at the ends of what the collocation takes: values that are not
finite, next to the largest number, and windows whose terms cancel over hundreds
of decades (the samples of a window's two halves are each other's negatives but
for one, by a few bits)."""
import numpy as np

KINDS = ("inf", "nan", "large", "wide", "cancel")


def faces(kind, nx, ny, ng, rng):
    w, h = nx + 2 * ng, ny + 2 * ng
    if kind in ("inf", "nan"):
        f = rng.normal(size=(h, w))
        f[rng.random((h, w)) < 0.05] = np.inf if kind == "inf" else np.nan
        if kind == "inf":
            f[rng.random((h, w)) < 0.05] = -np.inf
    elif kind == "large":
        f = rng.normal(size=(h, w)) * 1e300
    elif kind == "wide":
        f = rng.normal(size=(h, w)) * 10.0 ** rng.integers(-250, 250, (h, w))
    else:
        f = np.zeros((h, w))
        width = 2 * ng
        for j in range(h):
            half = rng.uniform(1, 2, ng) * np.sort(10.0 ** rng.uniform(-250, 290, ng))[::-1]
            row = np.concatenate([half, -half[::-1]])
            row[rng.integers(width)] *= 1 + rng.integers(-1, 2) * 2.0 ** -rng.integers(20, 53)
            f[j, rng.integers(0, w - width + 1):][:width] = row
    return f.ravel()


def both_axes(f, nx, ny, ng):
    """The rows' samples for axis 0, and the same windows along columns."""
    return f, np.ascontiguousarray(f.reshape(ny + 2 * ng, nx + 2 * ng).T).ravel()
