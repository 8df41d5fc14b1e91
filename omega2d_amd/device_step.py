"""Advection steps with every array resident in HBM: particles, optionally around one body.

This is the device-resident counterpart of the C++ host mirror (omega2d_amd/host/Convection.h
and host/BEM.h) for the gpu_hip environment. The mirror follows src/Convection.h:172-598 and
src/BEMHelper.h:43-260 on host arrays, as the reference's callers hold them. This module makes
the same calls in the same order on torch tensors. A step enqueues everything on torch's
current stream and copies nothing between host and device.

The body is a closed loop of panels attached to the ground, reactive and augmented (one
rotation unknown and the circulation constraint row, src/Coefficients.h:430-572), with one
(vortex) or two (vortex + source) unknowns per panel. Each stage of a step:
  * solves the boundary-element system: panel-centre velocities from the particles
    (points_affect_panels) plus the freestream, right-hand side -u.t (and -u.n), augmented row
    2 vol omega_error + reabsorbed circulation (src/BEMHelper.h:116-137, src/RHS.h:54-115);
  * sums particles on particles and panels on particles (src/Convection.h:172-223), with the
    solved rotation's strengths added to the panels (src/Surfaces.h:556-620) and the sums
    finalized as u = fs + u / (2 pi) (src/ElementBase.h:215-221);
  * moves the particles in fp64 (src/ElementBase.h:276-359) and pushes them out of the body's
    inner layer (clear_inner_layer, method 1, src/Reflect.h:733-762).
The matrix is assembled and LU-factored once; the body does not move.
"""
import math

import numpy as np
import torch

from . import device as dv

FACTOR = 0.5 / math.pi
CLEAR_CUTOFF = 0.5 / math.sqrt(2.0 * math.pi)  # layer thickness in particle spacings


def panel_bases(nx, ny, idx):
    """Unit tangents, normals (into the fluid) and lengths of each panel
    (src/Surfaces.h:699-724): t = (p1 - p0) * (1 / |p1 - p0|), n = (-t_y, t_x)."""
    a, c = idx[0::2].astype(np.int64), idx[1::2].astype(np.int64)
    t0, t1 = nx[c] - nx[a], ny[c] - ny[a]
    base = np.sqrt(t0 * t0 + t1 * t1)
    inv = 1.0 / base
    t0, t1 = t0 * inv, t1 * inv
    return t0, t1, -t1, t0, base


def geom_center(nx, ny, idx):
    """Signed area and centroid of the panel loop from the fan of triangles (origin, node j,
    node j+1), each by Heron's formula (src/Surfaces.h:623-677)."""
    asum = xsum = ysum = 0.0
    for j, jp1 in zip(idx[0::2].tolist(), idx[1::2].tolist()):
        x0, y0, x1, y1 = float(nx[j]), float(ny[j]), float(nx[jp1]), float(ny[jp1])
        xc, yc = (0.0 + x0 + x1) / 3.0, (0.0 + y0 + y1) / 3.0
        px, py = x1 - x0, y1 - y0
        a = math.sqrt(x0 * x0 + y0 * y0)
        b = math.sqrt(px * px + py * py)
        c = math.sqrt(x1 * x1 + y1 * y1)
        hs = 0.5 * (a + b + c)
        asq = hs * (hs - a) * (hs - b) * (hs - c)
        ar = math.sqrt(asq) if asq > 0.0 else 0.0
        if y0 * px - x0 * py < 0.0:
            ar = -ar
        asum += ar
        xsum += xc * ar
        ysum += yc * ar
    return asum, xsum / asum, ysum / asum


class Body:
    """A closed panel loop attached to the ground, reactive and augmented, on one device.

    nx, ny: node coordinates (float32 values, as the reference's ElementPacket<float> holds
    them); idx: two node indices per panel; nunk: 1 (vortex) or 2 (vortex + source) unknowns
    per panel."""

    def __init__(self, nx, ny, idx, nunk=1, device="cuda"):
        if nunk not in (1, 2):
            raise ValueError("nunk must be 1 or 2")
        nx = np.asarray(nx, dtype=np.float32).astype(np.float64)
        ny = np.asarray(ny, dtype=np.float32).astype(np.float64)
        idx = np.asarray(idx, dtype=np.uint32)
        self.np_, self.nunk = len(idx) // 2, nunk
        tx, ty, pnx, pny, area = panel_bases(nx, ny, idx)
        self.vol, cx, cy = geom_center(nx, ny, idx)
        a, c = idx[0::2].astype(np.int64), idx[1::2].astype(np.int64)
        # vector from the geometric centre to each panel centre (src/Surfaces.h:595-597)
        ddx = 0.5 * (nx[a] + nx[c]) - cx
        ddy = 0.5 * (ny[a] + ny[c]) - cy
        T = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(device)  # noqa: E731
        self.nx, self.ny = T(nx), T(ny)
        self.idx = torch.from_numpy(idx.astype(np.int32)).to(device)
        self.tx, self.ty, self.pnx, self.pny = T(tx), T(ty), T(pnx), T(pny)
        self.ddx, self.ddy = T(ddx), T(ddy)
        # the unit-rotation velocity at the panels (src/BEMHelper.h:203-210): the panels carry
        # the unit rotation's strengths and act on particles just off each panel's centre
        # (represent_as_particles, src/Surfaces.h:788-843, offset 1e-4, spacing = first length)
        rvs, rss = self.rot_strengths(torch.ones((), dtype=torch.float64, device=device))
        mx, my = self._offset_points(nx, ny, idx, pnx, pny, area)
        uu, uv = dv.panels_on_points(self.nx, self.ny, self.idx, rvs, rss, T(mx), T(my))
        uu, uv = uu[:self.np_] * FACTOR, uv[:self.np_] * FACTOR
        n = self.np_ * nunk + 1
        self.A = torch.empty((n, n), dtype=torch.float64, device=device)
        dv.bem_assemble(self.nx, self.ny, self.idx, nunk, True, uu.contiguous(),
                        uv.contiguous(), self.vol, out=self.A)
        dv.bem_factor(self.A)
        self.vs = torch.zeros(self.np_, dtype=torch.float64, device=device)
        self.ss = torch.zeros_like(self.vs)
        self.omega = torch.zeros((), dtype=torch.float64, device=device)
        self.omega_error = torch.zeros((), dtype=torch.float64, device=device)
        self.reabsorbed = torch.zeros((), dtype=torch.float64, device=device)

    @staticmethod
    def _offset_points(nx, ny, idx, pnx, pny, area):
        px, py = [], []
        ips = area[0]
        for i, (a, c) in enumerate(zip(idx[0::2].tolist(), idx[1::2].tolist())):
            nshed = 1 + max(0, int(area[i] / (1.2 * ips)))
            for j in range(nshed):
                wgt = (1 + 2 * j) / (2 * nshed)
                px.append(wgt * nx[c] + (1.0 - wgt) * nx[a] + 0.0001 * pnx[i])
                py.append(wgt * ny[c] + (1.0 - wgt) * ny[a] + 0.0001 * pny[i])
        f = lambda v: np.asarray(v, dtype=np.float64).astype(np.float32).astype(np.float64)  # noqa
        return f(px), f(py)

    def rot_strengths(self, rotvel):
        """Vortex and source strengths of a solid-body rotation rotvel about the geometric
        centre (src/Surfaces.h:570-620)."""
        ui = -rotvel * self.ddy
        vi = rotvel * self.ddx
        return (-1.0 * (ui * self.tx + vi * self.ty), -1.0 * (ui * self.ty - vi * self.tx))

    def _scalar(self, v):
        return torch.as_tensor(v, dtype=torch.float64, device=self.tx.device).reshape(())

    def solve(self, x, y, s, fs):
        """The boundary-element solve for particles (x, y, s) and freestream fs."""
        pu, pv = torch.zeros((2, self.np_), dtype=torch.float64, device=x.device)
        dv.points_on_panels(x, y, s, self.nx, self.ny, self.idx, pu=pu, pv=pv)
        rhs = dv.body_rhs(pu, pv, fs, FACTOR, self.tx, self.ty, self.pnx, self.pny, self.nunk,
                          self._scalar(self.reabsorbed), 2.0 * self.vol,
                          self._scalar(self.omega_error))
        sol = dv.bem_solve(rhs, torch.empty_like(rhs))
        self.vs, self.ss, self.omega, self.omega_error = dv.body_unpack(sol, self.nunk)

    def add_vels(self, x, y, u, v):
        """Panels (with the solved rotation's strengths) on points, added into u, v."""
        vs, ss = dv.body_strengths(self.vs.contiguous(), self.ss.contiguous(),
                                   self._scalar(self.omega), self.tx, self.ty, self.ddx, self.ddy)
        dv.panels_on_points(self.nx, self.ny, self.idx, vs, ss, x, y, tu=u, tv=v)

    def clear(self, x, y, s, r, ips):
        """Push particles out of the inner layer (method 1), in place."""
        circ, _ = dv.clear_inner(1, self.nx, self.ny, self.idx, self.pnx, self.pny,
                                 CLEAR_CUTOFF, ips, x, y, s, r)
        self.reabsorbed = self.reabsorbed + circ[0]


class Stepper:
    """Euler, Ralston RK2 or Ralston RK3 steps of particles (x, y, s, r: float64 device tensors,
    updated in place) with the given core and precision form, optionally around one Body."""

    def __init__(self, x, y, s, r, *, core="v2", precision="split", fs=(0.0, 0.0), body=None,
                 ips=0.01):
        self.x, self.y, self.s, self.r = x, y, s, r
        self.core, self.precision, self.fs = core, precision, (float(fs[0]), float(fs[1]))
        self.body, self.ips = body, float(ips)
        self.stages = []

    def vels(self, x, y):
        """Finalized velocities of the particles at (x, y) (src/Convection.h:172-243)."""
        if self.body is not None:
            self.body.solve(x, y, self.s, self.fs)
        u, v = torch.zeros((2, *x.shape), dtype=x.dtype, device=x.device)
        dv.points_on_points(x, y, self.s, self.r, x, y, self.r, core=self.core,
                            precision=self.precision, tu=u, tv=v)
        if self.body is not None:
            self.body.add_vels(x, y, u, v)
        return dv.finalize(u, v, self.fs, FACTOR)

    def _clear(self, x, y):
        if self.body is not None:
            self.body.clear(x, y, self.s, self.r, self.ips)

    def _moved(self, dt, w, us, vs):
        x, y = dv.rk_advance(self.x, self.y, us, vs, w, dt)
        self._clear(x, y)
        return x, y

    def _combined(self, dt, w, us, vs):
        _, _, u, v = dv.rk_advance(self.x, self.y, us, vs, w, dt, self.x, self.y, combined=True)
        self._clear(self.x, self.y)
        return u, v

    def step(self, dt, order=2):
        """One step of the given order (src/Convection.h:274-303, 390-466, 472-598). Returns
        the velocity the reference leaves in the particles (the stage combination for orders
        2 and 3, computed as the position update combines them); self.stages holds the stage
        velocities."""
        if order == 1:
            u0, v0 = self.vels(self.x, self.y)
            self.stages = [(u0, v0)]
            dv.rk_move(self.x, self.y, [u0], [v0], [1.0], dt)
            self._clear(self.x, self.y)
            return u0, v0
        if order == 2:
            u0, v0 = self.vels(self.x, self.y)
            x1, y1 = self._moved(2.0 / 3.0 * dt, [1.0], [u0], [v0])
            u1, v1 = self.vels(x1, y1)
            self.stages = [(u0, v0), (u1, v1)]
            w = [0.25, 0.75]
            return self._combined(dt, w, [u0, u1], [v0, v1])
        if order == 3:
            u0, v0 = self.vels(self.x, self.y)
            x1, y1 = self._moved(0.5 * dt, [1.0], [u0], [v0])
            u1, v1 = self.vels(x1, y1)
            x2, y2 = self._moved(0.75 * dt, [1.0], [u1], [v1])
            u2, v2 = self.vels(x2, y2)
            self.stages = [(u0, v0), (u1, v1), (u2, v2)]
            w = [2.0 / 9.0, 3.0 / 9.0, 4.0 / 9.0]
            return self._combined(dt, w, [u0, u1, u2], [v0, v1, v2])
        raise ValueError("order must be 1, 2 or 3")
