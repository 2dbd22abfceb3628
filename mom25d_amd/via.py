"""Via (vertical wire) kernels on the device (src/mom25d/via.py:127-235).

A via's current is constant along each chain (the layers between two interfaces where it touches metal); its end
charges spread over the fan triangles around the via vertex and enter through G_q like the strips' charges. Per
frequency, one m25x_spectra launch gives every spectrum the vias need on the frequency's contour:
  D(k, span)   the smooth via -> interface kernel of a chain span seen on interface k, tabulated on the uniform
               grid (one Hankel transform and one spline product for all of them)
  R(sm, sn)    the via -> via reaction remainder between two spans, transformed at the pairs' distances (or
               tabulated, for many pairs)
and homog() the analytic K0 part of the reaction, on the host.
"""
import numpy as np
import torch
from scipy.special import kv

from .base import C0, MU0
from . import _lib as L
from . import device as dv
from .multilayer import (NFINE, NRHO, Requests, _blank_tables, _request_tables, _set_tables, device_contour, hankel,
                         quad_grid, spline_operator)

NRHO_VIA = 200                    # the quadratic grid of the via kernels' tables


class DevTable1D:
    """A radial table on the uniform grid of nfine points (values on the device), linear lookup (via.py:111-123)."""

    def __init__(self, v, rho_max, nfine=NFINE):
        self.v, self.rho_max, self.nfine = v, rho_max, nfine
        self._dr = np.linspace(0, rho_max, nfine)[1]

    def __call__(self, r):
        v = self.v.cpu().numpy()
        u = np.minimum(np.asarray(r) / self._dr, self.nfine - 1.000001)
        i = u.astype(np.int64)
        t = u - i
        return v[i] * (1 - t) + v[i + 1] * t


def span_layers(span):
    """The dielectric layers a chain from interface span[0] up to span[1] runs through."""
    return range(span[0] + 1, span[1] + 1)


def homog(st, w, sm, sn, rho):
    """The analytic part of the reaction of two spans through their shared layers j: a line current in the
    homogeneous medium of layer j, (j w mu0 h_j / 2 pi) K0(j k_j rho), k_j with Im k_j <= 0 (host)."""
    rho = np.atleast_1d(np.asarray(rho, float))
    out = np.zeros(rho.shape, complex)
    k0sq = (w / C0) ** 2
    for j in sorted(set(span_layers(sm)) & set(span_layers(sn))):
        kj = np.sqrt(k0sq * st.eps(j) + 0j)
        kj = -kj if kj.imag > 0 else kj
        out += 1j * w * MU0 * st.layers[j - 1].h / (2 * np.pi) * kv(0, 1j * kj * rho)
    return out


def point_distances(rho_max, groups):
    """The distances of point_kernels' transforms, on the device (fixed by the mesh): the tables' grid, the via tables'
    grid and each span pair's chain distances, in order."""
    return dv.on_dev(np.concatenate([quad_grid(rho_max, NRHO), quad_grid(rho_max, NRHO_VIA)] +
                                    [dd for _, _, dd in groups.values()]), dv.f64)


def point_kernels(f, stack, layers, rho_max, dmax, spans, groups, rho):
    """(tables, D, R) of a frequency: green_tables's tables, the via -> interface kernels D (a row of NFINE points per
    span and interface) and the via -> via reactions R at the distances of groups {(span, span): (m, n, distances)}, in
    order. One contour, one spectra launch, one Hankel launch and one spline launch per grid for all of them; the
    separate classes would take three of each and a read-back. rho: point_distances of the same groups."""
    st, w = stack.at(f), 2 * np.pi * f
    contour = device_contour(f, stack, rho_max)
    tables = _blank_tables(f, st, w, layers, dmax)
    tabs, req = list(tables.values()), Requests()
    _request_tables(req, tabs)
    nt = req.rows
    for lo, hi in spans:
        for k in layers:
            req.add(L.SPEC_VIA_D, (k, lo, hi))
    nd = req.rows - nt
    sets = [(NRHO, 0, nt), (NRHO_VIA, nt, nd)]
    for (sm, sn), (_, _, dd) in groups.items():
        sets.append((len(dd), req.add(L.SPEC_VIA_R, (sm[0], sm[1], sn[0], sn[1])), 1))
    W = req.run(st, w, contour)
    out = dv.hankel_sets(rho, sets, contour[0], W, 2 * np.pi)
    _set_tables(tabs, out[0], contour, rho_max, NRHO, NFINE)
    D = dv.resample(spline_operator(NRHO_VIA, NFINE), out[1])
    R = torch.cat([x[0] for x in out[2:]]) if len(out) > 3 else out[2][0]
    return tables, D, R


class ViaKernels:
    """Per-frequency via kernels for chain spans [(k_bot, k_top), ...] and the metal interfaces (via.py:179-235)."""

    def __init__(self, f, stack, spans, interfaces, rho_max, nrho=NRHO_VIA):
        self.f, self.w = f, 2 * np.pi * f
        self.st = stack.at(f)
        self.contour = device_contour(f, stack, rho_max)
        self.rho_max, self.nrho, self.D = rho_max, nrho, {}
        self.spans = sorted(set(spans))
        req, d_rows, self._r_rows = Requests(), [], {}
        for span in self.spans:
            for k in interfaces:
                d_rows.append(((k, span), req.add(L.SPEC_VIA_D, (k, span[0], span[1]))))
        for sm in self.spans:
            for sn in self.spans:
                self._r_rows[(sm, sn)] = req.add(L.SPEC_VIA_R, (sm[0], sm[1], sn[0], sn[1]))
        self._W = req.run(self.st, self.w, self.contour)
        if d_rows:
            grid = dv.on_dev(quad_grid(rho_max, nrho), dv.f64)      # the D rows come first in W
            fine = dv.resample(spline_operator(nrho, NFINE), hankel(self._W[:len(d_rows)], self.contour, grid))
            for j, (key, _) in enumerate(d_rows):
                self.D[key] = DevTable1D(fine[j], rho_max)

    def _r_row(self, sm, sn):
        row = self._r_rows.get((tuple(sm), tuple(sn)))
        if row is None:
            raise KeyError(f"no via reaction between spans {sm} and {sn} at this frequency")
        return self._W[row:row + 1]

    def R(self, sm, sn, rho):
        """The via-via reaction remainder at distances rho (host array in, host array out)."""
        rho = np.atleast_1d(np.asarray(rho, float))
        return hankel(self._r_row(sm, sn), self.contour, dv.on_dev(rho, dv.f64))[0].cpu().numpy()

    def R_table(self, sm, sn):
        """R tabulated on the uniform grid (one transform on the quadratic grid): for many pairs of one span pair."""
        grid = dv.on_dev(quad_grid(self.rho_max, self.nrho), dv.f64)
        vals = hankel(self._r_row(sm, sn), self.contour, grid)
        return DevTable1D(dv.resample(spline_operator(self.nrho, NFINE), vals)[0], self.rho_max)

    def homog(self, sm, sn, rho):
        """The analytic part of the reaction of two spans (host)."""
        return homog(self.st, self.w, sm, sn, rho)
