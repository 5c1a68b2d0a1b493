"""Trajectory simulator (counterpart of clode/trajectory.py).

Stores the initial point and every nout-th step, up to max_store samples per
member, and returns one ``TrajectoryOutput`` per member with the stored part
only (clode/trajectory.py:18-266).
"""
from __future__ import annotations

from functools import lru_cache
from typing import Any, Callable, Dict, List, Optional, Tuple, Union

import numpy as np
from numpy.lib import recfunctions as rfn

from .cpp.clode_cpp_wrapper import SolverParams, TrajectorySimulatorBase, member_rows
from .runtime import CLDeviceType, CLVendor, _clode_root_dir
from .solver import Simulator, Stepper


@lru_cache(maxsize=256)
def _fields(names: Tuple[str, ...]) -> np.dtype:
    return np.dtype({"names": list(names), "formats": [np.float64] * len(names)})


def _struct(names: List[str]) -> np.dtype:
    """A row of doubles with these names: the same object for the same names, which compares fastest."""
    return _fields(tuple(names))


class TrajectoryOutput:
    def __init__(self, t: np.ndarray, x: np.ndarray, dx: np.ndarray, aux: np.ndarray, variable_names: List[str],
                 aux_names: List[str]) -> None:
        self.t = t
        xdt = _struct(variable_names)
        self.x = rfn.unstructured_to_structured(np.ascontiguousarray(x), dtype=xdt)
        self.dx = rfn.unstructured_to_structured(np.ascontiguousarray(dx), dtype=xdt)
        if len(aux_names) > 0:
            self.aux = rfn.unstructured_to_structured(np.ascontiguousarray(aux), dtype=_struct(aux_names))
        self._variable_names = variable_names
        self._aux_names = aux_names

    @classmethod
    def _of_structured(cls, t: np.ndarray, x: np.ndarray, dx: np.ndarray, aux: Optional[np.ndarray],
                       variable_names: List[str], aux_names: List[str]) -> "TrajectoryOutput":
        """From arrays that are structured already (one member's rows of the ensemble's arrays)."""
        out = cls.__new__(cls)
        out.t, out.x, out.dx = t, x, dx
        if aux is not None:
            out.aux = aux
        out._variable_names, out._aux_names = variable_names, aux_names
        return out

    def __repr__(self) -> str:
        return (f"TrajectoryOutput( length: {len(self.t)}, variable names: {self._variable_names}, "
                f"aux variable names: {self._aux_names} )")

    def to_ndarray(self, slot: str, **kwargs) -> np.ndarray:
        a = getattr(self, slot)
        names = a.dtype.names
        if not kwargs and names is not None and a.dtype == _fields(names) and a.flags.c_contiguous:
            # fields of double, one after the other: the same memory as columns
            return a.view(np.float64).reshape(a.shape + (len(names),))
        return rfn.structured_to_unstructured(a, **kwargs)


class TrajectorySimulator(Simulator):
    """Simulator that stores trajectories."""

    _integrator: TrajectorySimulatorBase

    def __init__(
        self,
        variables: Dict[str, float],
        parameters: Dict[str, float],
        aux: Optional[List[str]] = None,
        num_noise: int = 0,
        src_file: Optional[str] = None,
        rhs_equation: Optional[Callable] = None,
        supplementary_equations: Optional[List[Callable[[Any], Any]]] = None,
        stepper: Stepper = Stepper.rk4,
        dt: float = 0.1,
        dtmax: float = 1.0,
        abstol: float = 1e-6,
        reltol: float = 1e-4,
        max_steps: int = 1000000,
        max_store: int = 1000000,
        nout: int = 1,
        solver_parameters: Optional[SolverParams] = None,
        t_span: Tuple[float, float] = (0.0, 1000.0),
        single_precision: Union[bool, str] = True,
        device_type: Optional[CLDeviceType] = None,
        vendor: Optional[CLVendor] = None,
        platform_id: Optional[int] = None,
        device_id: Optional[int] = None,
        device_ids: Optional[List[int]] = None,
    ) -> None:
        super().__init__(variables=variables, parameters=parameters, aux=aux, num_noise=num_noise,
                         src_file=src_file, rhs_equation=rhs_equation,
                         supplementary_equations=supplementary_equations, stepper=stepper, dt=dt, dtmax=dtmax,
                         abstol=abstol, reltol=reltol, max_steps=max_steps, max_store=max_store, nout=nout,
                         solver_parameters=solver_parameters, t_span=t_span, single_precision=single_precision,
                         device_type=device_type, vendor=vendor, platform_id=platform_id, device_id=device_id,
                         device_ids=device_ids)
        self._device_t = self._device_x = self._device_dx = self._device_aux = None

    def _create_integrator(self) -> None:
        self._integrator = TrajectorySimulatorBase(self._pi, self._stepper.value, self._single_precision,
                                                   self._runtime, _clode_root_dir)

    def trajectory(self, t_span: Optional[Tuple[float, float]] = None, update_x0: bool = True,
                   fetch_results: bool = True):
        """Integrate and store trajectories; optionally return them."""
        if t_span is not None:
            self.set_tspan(t_span=t_span)
        self._integrator.trajectory()
        self._device_t = self._device_x = self._device_dx = self._device_aux = None
        self._device_final_state = self._device_dt = self._device_tf = None
        if update_x0:
            self._integrator.shift_x0()
            self._device_initial_state = None
        if fetch_results:
            return self.get_trajectory()
        return None

    def get_trajectory(self):
        store = self._sp.max_store
        n = self._ensemble_size
        # every member's samples are rows of one array per kind, transposed to
        # that order on the device; each output has a copy of its own rows
        t = self._integrator.get_t_members()
        if t.shape[1] < store:
            raise ValueError(f"{t.shape[1]} samples per member are stored, max_store is {store}")
        x, dx, aux = (get() for get in (self._integrator.get_x_members, self._integrator.get_dx_members,
                                        self._integrator.get_aux_members))
        self._device_t = t[:, :store]
        self._device_x, self._device_dx, self._device_aux = (a.transpose(0, 2, 1)[:, :, :store] for a in (x, dx, aux))
        names, aux_names = self.variable_names, self.aux_names
        counts = np.minimum(np.array(self._integrator.get_n_stored()) + 1, store).tolist()
        make = TrajectoryOutput._of_structured
        if n == 1:  # its rows are the arrays' first
            k = counts[0]
            return make(t[0, :k], x.view(_struct(names))[0, :k, 0], dx.view(_struct(names))[0, :k, 0],
                        aux.view(_struct(aux_names))[0, :k, 0] if len(aux_names) > 0 else None, names, aux_names)
        ts = member_rows(t, counts, np.dtype(np.float64))
        xs, dxs = (member_rows(a, counts, _struct(names)) for a in (x, dx))
        auxs = member_rows(aux, counts, _struct(aux_names)) if len(aux_names) > 0 else [None] * n
        return [make(*member, names, aux_names) for member in zip(ts, xs, dxs, auxs)]
