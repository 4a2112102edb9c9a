"""Initial position / velocity distributions (distributions.py:12-185 of the reference).

``draw(n)`` is the reference's host draw (scipy.stats on numpy's global RNG), so a seeded run
replays the reference's inputs exactly.  ``draw_device(n, seed)`` (Gaussian families) draws on the
GPU with Philox4x32-10 + Box-Muller into device buffers, for runs too large to ship from the host.
"""
from __future__ import annotations

from abc import ABC, abstractmethod
from dataclasses import dataclass
from pathlib import Path

import numpy as np
from scipy.stats import norm, uniform


class Distribution(ABC):
    @abstractmethod
    def draw(self, n: int) -> np.ndarray:
        """n samples as a (3, n) float64 array."""

    def save_to_hdf(self, filepath: Path, run_name: str):
        from .hdf import save_distribution

        save_distribution(self, filepath, run_name)

    # device forms: (mean[3], sigma[3]) of independent Gaussians, or None if not Gaussian
    def gaussian_params(self):
        return None

    # (radius, z) of a uniform disc at fixed z, or None if not such a disc
    def disc_params(self):
        return None

    def draw_device(self, n: int, seed: int, offset: int = 0, ctx=None, out=None):
        """Draw n samples on the device from the counter-based streams of key ``seed`` (molecule
        index + ``offset`` as the counter, so any chunking of a run draws the same molecules);
        returns three DeviceArrays (rows of draw(n); ``out``, three arrays of at least n, to fill
        existing ones).  The values follow the distribution, not the host draw's numpy sequence."""
        from .device import get_context
        from .engine import draw_disc, draw_gaussian

        p = self.gaussian_params()
        if p is not None:
            mean, sigma = p
            return draw_gaussian(ctx or get_context(), n, mean, sigma, seed, offset, out=out)
        q = self.disc_params()
        if q is not None:
            radius, z = q
            return draw_disc(ctx or get_context(), n, radius, z, seed, offset, out=out)
        raise NotImplementedError(f"{type(self).__name__} has no device sampler")


def _plain(*values) -> bool:
    return all(type(v) in (int, float, np.float64) for v in values)


def _normals(loc, scale, n: int) -> np.ndarray:
    """norm.rvs(loc, scale, n): for plain numbers its own two operations on the same random state, without the
    argument handling that made up nearly all of a short draw's time (17 us)."""
    if _plain(loc, scale) and scale > 0 and type(n) is int:
        return norm.random_state.standard_normal(n) * scale + loc
    return norm.rvs(loc=loc, scale=scale, size=n)


def _uniforms(n: int) -> np.ndarray:
    """uniform.rvs(size=n) (on [0, 1)), likewise."""
    if type(n) is int:
        return uniform.random_state.uniform(0.0, 1.0, n)
    return uniform.rvs(size=n)


@dataclass
class GaussianDistribution(Distribution):
    mean: float
    sigma: float

    def __post_init__(self):
        self.dist = norm

    def draw(self, n: int) -> np.ndarray:
        if self.dist is norm:
            return _normals(self.mean, self.sigma, n)
        return self.dist.rvs(loc=self.mean, scale=self.sigma, size=n)

    def plot(self):
        import matplotlib.pyplot as plt

        fig, ax = plt.subplots()
        x = self.mean + np.linspace(-5, 5, 1000) * self.sigma
        ax.plot(x, self.dist.pdf(x, loc=self.mean, scale=self.sigma))

    def save_to_hdf(self, filepath: Path, run_name: str, group_name: str = ""):
        raise NotImplementedError("Saving GaussianDistribution to hdf is not implemented. Save child class instead.")


@dataclass
class CeNTREXVelocityDistribution(Distribution):
    """Independent Gaussians along X, Y, Z; draw order vx, vy, vz (distributions.py:69-76)."""

    vx: float = 0.0
    sigmax: float = 39.5
    vy: float = 0.0
    sigmay: float = 39.5
    vz: float = 184.0
    sigmaz: float = 16.0

    def draw(self, n: int) -> np.ndarray:
        return np.array((GaussianDistribution(self.vx, self.sigmax).draw(n),
                         GaussianDistribution(self.vy, self.sigmay).draw(n),
                         GaussianDistribution(self.vz, self.sigmaz).draw(n)))

    def gaussian_params(self):
        return (np.array([self.vx, self.vy, self.vz], float), np.array([self.sigmax, self.sigmay, self.sigmaz], float))


@dataclass
class CeNTREXPositionDistribution(Distribution):
    """Uniform disc of diameter d at z (distributions.py:112-119): theta then sqrt(u)."""

    d: float = 0.02
    z: float = 0.25 * 0.0254

    def draw(self, n: int) -> np.ndarray:
        theta = _uniforms(n) * 2 * np.pi
        r = np.sqrt(_uniforms(n)) * self.d / 2
        return np.array((r * np.cos(theta), r * np.sin(theta), np.full(n, self.z)))

    def disc_params(self):
        return (self.d / 2, float(self.z))


@dataclass
class GaussianPositionDistribution(Distribution):
    """Gaussian x, y at fixed z; draw order x, y (distributions.py:155-162)."""

    sigmax: float = 0.25 * 25.4 / 5 * 3.8e-3
    sigmay: float = 0.25 * 25.4 / 5 * 3.8e-3
    z: float = 0.25 * 0.0254

    def draw(self, n: int) -> np.ndarray:
        x = GaussianDistribution(0, self.sigmax).draw(n)
        y = GaussianDistribution(0, self.sigmay).draw(n)
        return np.vstack((x, y, np.full(n, self.z)))

    def gaussian_params(self):
        return (np.array([0.0, 0.0, self.z], float), np.array([self.sigmax, self.sigmay, 0.0], float))


def draw_chunks(xdist: Distribution, vdist: Distribution, n: int, chunks: int) -> tuple[np.ndarray, np.ndarray]:
    """``chunks`` times vdist.draw(n) then xdist.draw(n) (trajectory_simulator.py:52-60 of the reference), joined:
    X and V of shape (3, chunks n).

    The reference's distributions draw from one random state, whose normal stream does not depend on how it is cut
    into calls: with Gaussian velocities and either position distribution, a chunk's normals are one call and
    its uniforms another, and the arithmetic is done once on all chunks, element for element the same."""
    total = n * chunks
    replaced = any("draw" in getattr(d, "__dict__", ()) for d in (xdist, vdist))  # on the instance
    if not replaced and min(n, chunks) > 0 and type(vdist) is CeNTREXVelocityDistribution \
            and norm.random_state is uniform.random_state:
        vp = (vdist.vx, vdist.sigmax, vdist.vy, vdist.sigmay, vdist.vz, vdist.sigmaz)
        if _plain(*vp) and all(s > 0 for s in vp[1::2]):  # NaN is refused by the plain draws below
            rs = norm.random_state
            if type(xdist) is GaussianPositionDistribution and _plain(xdist.sigmax, xdist.sigmay, xdist.z) \
                    and xdist.sigmax > 0 and xdist.sigmay > 0:
                g = rs.standard_normal(5 * total).reshape(chunks, 5, n)
                X = np.stack([(g[:, 3] * xdist.sigmax + 0).reshape(-1), (g[:, 4] * xdist.sigmay + 0).reshape(-1),
                              np.full(total, xdist.z, dtype=np.float64)])
            elif type(xdist) is CeNTREXPositionDistribution and _plain(xdist.d, xdist.z):
                g, u = np.empty((chunks, 3, n)), np.empty((chunks, 2, n))
                for c in range(chunks):
                    g[c] = rs.standard_normal(3 * n).reshape(3, n)
                    u[c] = rs.uniform(0.0, 1.0, 2 * n).reshape(2, n)
                theta = u[:, 0].reshape(-1) * 2 * np.pi
                r = np.sqrt(u[:, 1].reshape(-1)) * xdist.d / 2
                X = np.stack([r * np.cos(theta), r * np.sin(theta), np.full(total, xdist.z, dtype=np.float64)])
            else:
                g = None
            if g is not None:
                V = np.stack([(g[:, k] * vp[2 * k + 1] + vp[2 * k]).reshape(-1) for k in range(3)])
                return X, V
    vs, xs = [], []
    for _ in range(chunks):
        vs.append(np.asarray(vdist.draw(n), dtype=np.float64).reshape(3, n))
        xs.append(np.asarray(xdist.draw(n), dtype=np.float64).reshape(3, n))
    if not vs:
        return np.zeros((3, 0)), np.zeros((3, 0))
    return np.concatenate(xs, axis=1), np.concatenate(vs, axis=1)
