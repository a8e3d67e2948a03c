"""Free energy, currents, field and superfluid density
(svirl/observables/observables.py) on libglx kernels."""
import ctypes

import numpy as np

from svirl_amd import _native as nat


class Observables:
    def __init__(self, par, mesh, vars, params):
        self.par = par
        self.mesh = mesh
        self.vars = vars
        self.params = params
        self.cfg = par.cfg
        self._edge2 = None  # second link-sized buffer for the fused pass

    def _grid(self):
        c = self.cfg
        return nat.Grid(int(c.Nx), int(c.Ny), float(c.dx), float(c.dy))

    def _sync_device(self):
        self.vars._psi.sync_d()
        self.vars._vp.sync_d()
        if self.params._vpei is not None:
            self.params._vpei.sync_d()

    @property
    def superfluid_density(self):
        """|psi|^2 on nodes (observables.py:29-33)."""
        self.vars._psi.sync_d()
        psi = self.vars._psi.get_h()
        return np.square(psi.real) + np.square(psi.imag)

    @property
    def magnetic_field(self):
        """B per cell from abei + ab (observables.py:36-58)."""
        self._sync_device()
        out = self.vars._tmp_cell_var_h()
        self._cols(out, None, None)
        return self._cells(out)

    def _cols(self, B, J, Js):
        """B, J and J_s of the state into device arrays (None: not), each
        in column order: [i, j] of the host arrays."""
        p = self.params
        nat.call("glx_bulk_observables_cols", self.par.prec, self._grid(),
                 float(p.gl_parameter_squared_h()) if p.solveA else 0.0, float(p.homogeneous_external_field),
                 nat.ptr(self.mesh.material_tiling_h()), self.vars.order_parameter_h().ptr,
                 nat.ptr(p.external_irregular_vector_potential_h()), nat.ptr(self.vars.vector_potential_h()),
                 nat.ptr(B), nat.ptr(J), nat.ptr(Js))

    def _host(self, dev, first, shape):
        out = np.empty(shape, dtype=dev.dtype)
        nat.call("glx_memcpy_d2h", out.ctypes.data, dev.ptr + int(first) * dev.dtype.itemsize, out.nbytes)
        return out

    def _cells(self, dev):
        return self._host(dev, 0, (int(self.cfg.Nxc), int(self.cfg.Nyc)))

    def _edge_pair(self, dev):
        c = self.cfg
        return self._host(dev, 0, (int(c.Nxa), int(c.Nya))), self._host(dev, c.Na, (int(c.Nxb), int(c.Nyb)))

    @property
    def supercurrent_density(self):
        """J_s on links (observables.py:61-83)."""
        self._sync_device()
        out = self.vars._tmp_edge_var_h()
        self._cols(None, None, out)
        return self._edge_pair(out)

    @property
    def current_density(self):
        """kappa^2 (curl B - H) on links; J_s when kappa = inf
        (observables.py:86-110)."""
        if not self.params.solveA:
            return self.supercurrent_density
        self._sync_device()
        out = self.vars._tmp_edge_var_h()
        self._cols(None, out, None)
        return self._edge_pair(out)

    @property
    def normalcurrent_density(self):
        """J - J_s on links (observables.py:113-121); with A solved, J and
        J_s come from one fused pass (glx_bulk_observables_cols)."""
        if not self.params.solveA:
            jx, jy = self.current_density
            jsx, jsy = self.supercurrent_density
            return jx - jsx, jy - jsy
        _, (jx, jy), (jsx, jsy) = self._bulk(False)
        return jx - jsx, jy - jsy

    def bulk_observables(self):
        """(B, (Jx, Jy), (Jsx, Jsy)) as magnetic_field, current_density and
        supercurrent_density return them, from one pass over the nodes."""
        return self._bulk(True)

    def _bulk(self, want_B):
        self._sync_device()
        c = self.cfg
        p = self.params
        if self._edge2 is None:
            self._edge2 = nat.DeviceArray(int(c.Na + c.Nb), c.dtype)
        B = self.vars._tmp_cell_var_h() if want_B else None
        J = self.vars._tmp_edge_var_h() if p.solveA else None
        Js = self._edge2
        self._cols(B, J, Js)
        Bh = self._cells(B) if want_B else None
        js = self._edge_pair(Js)
        # J = J_s when kappa = inf (observables.py:86-110)
        jj = self._edge_pair(J) if J is not None else (js[0].copy(), js[1].copy())
        return Bh, jj, js

    @property
    def free_energy(self):
        """Total GL free energy (observables.py:124-149), FP64 accumulation."""
        self._sync_device()
        F = ctypes.c_double()
        p = self.params
        nat.call("glx_free_energy", self.par.prec, self._grid(), float(p.gl_parameter_squared_h()),
                 float(p.linear_coefficient_scalar_h()), nat.ptr(p.linear_coefficient_h()),
                 float(p.homogeneous_external_field), nat.ptr(self.mesh.material_tiling_h()),
                 self.vars.order_parameter_h().ptr, nat.ptr(p.external_irregular_vector_potential_h()),
                 nat.ptr(self.vars.vector_potential_h()), ctypes.byref(F))
        return self.cfg.dtype(F.value)

    def free_energy_fp64(self):
        """The same total as a Python float, without the cast to cfg.dtype."""
        self._sync_device()
        F = ctypes.c_double()
        p = self.params
        nat.call("glx_free_energy", self.par.prec, self._grid(), float(p.gl_parameter_squared_h()),
                 float(p.linear_coefficient_scalar_h()), nat.ptr(p.linear_coefficient_h()),
                 float(p.homogeneous_external_field), nat.ptr(self.mesh.material_tiling_h()),
                 self.vars.order_parameter_h().ptr, nat.ptr(p.external_irregular_vector_potential_h()),
                 nat.ptr(self.vars.vector_potential_h()), ctypes.byref(F))
        return F.value
