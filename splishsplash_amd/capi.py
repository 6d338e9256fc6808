"""ctypes binding of libsph_amd.so (the C-ABI of include/sph_capi.h).

`NeighborhoodSearch` mirrors CompactNSearch::NeighborhoodSearch as the
reference uses it (SPlisHSPlasH/NeighborhoodSearch.h, Simulation.cpp), and
`TimeStepDFSPH` mirrors SPH::TimeStepDFSPH plus the per-particle state it
steps. There is no fallback: if the library is missing, loading raises, and
if no gfx950 device is visible every compute call raises SPHError.
"""
import ctypes as C
import os

import numpy as np

from .params import DFSPHCounters, DFSPHParams, Emitter, FIELD_COMPONENTS, STAGES, default_params

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libsph_amd.so")

SPH_F32, SPH_F64 = 0, 1
_ERRORS = {-1: "invalid argument", -2: "HIP error", -3: "out of memory", -4: "invalid state",
           -5: "no gfx950 device", -6: "unknown field", -7: "size out of range"}


class SPHError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"{_ERRORS.get(code, code)}: {msg}")
        self.code = code


_lib = None
_up = C.POINTER(C.c_uint)
_fp = C.POINTER(C.c_float)
_dp = C.POINTER(C.c_double)
_szp = C.POINTER(C.c_size_t)
_vp = C.c_void_p

_SIGS = {
    "sph_last_error": (C.c_char_p, []),
    "sph_version": (C.c_int, []),
    "sph_device_count": (C.c_int, [C.POINTER(C.c_int)]),
    "sph_device_synchronize": (C.c_int, []),
    "sph_ns_create": (C.c_int, [C.c_double, C.c_int, C.POINTER(_vp)]),
    "sph_ns_destroy": (C.c_int, [_vp]),
    "sph_ns_set_radius": (C.c_int, [_vp, C.c_double]),
    "sph_ns_get_radius": (C.c_int, [_vp, _dp]),
    "sph_ns_reset": (C.c_int, [_vp]),
    "sph_ns_add_point_set": (C.c_int, [_vp, _vp, C.c_size_t, C.c_int, C.c_int, C.c_int, C.c_int, _vp, _up]),
    "sph_ns_resize_point_set": (C.c_int, [_vp, C.c_uint, _vp, C.c_size_t]),
    "sph_ns_update_point_sets": (C.c_int, [_vp]),
    "sph_ns_find_neighbors": (C.c_int, [_vp, C.c_int]),
    "sph_ns_find_neighbors_noalloc": (C.c_int, [_vp, C.c_size_t, C.c_double, _vp, _vp, C.c_size_t, _szp, _vp]),
    "sph_ns_query_point": (C.c_int, [_vp, _dp, C.c_uint, _up, C.c_uint, _up]),
    "sph_ns_z_sort": (C.c_int, [_vp]),
    "sph_ns_sort_field": (C.c_int, [_vp, C.c_uint, _vp, C.c_size_t]),
    "sph_ns_set_active_all": (C.c_int, [_vp, C.c_int]),
    "sph_ns_set_active_set": (C.c_int, [_vp, C.c_uint, C.c_int, C.c_int]),
    "sph_ns_set_active_pair": (C.c_int, [_vp, C.c_uint, C.c_uint, C.c_int]),
    "sph_ns_is_active_pair": (C.c_int, [_vp, C.c_uint, C.c_uint, C.POINTER(C.c_int)]),
    "sph_ns_n_point_sets": (C.c_int, [_vp, _up]),
    "sph_ns_n_points": (C.c_int, [_vp, C.c_uint, _szp]),
    "sph_ns_user_data": (C.c_int, [_vp, C.c_uint, C.POINTER(_vp)]),
    "sph_ns_n_neighbors": (C.c_int, [_vp, C.c_uint, C.c_uint, C.c_uint, _up]),
    "sph_ns_neighbor": (C.c_int, [_vp, C.c_uint, C.c_uint, C.c_uint, C.c_uint, _up]),
    "sph_ns_neighbor_list": (C.c_int, [_vp, C.c_uint, C.c_uint, C.c_uint, C.POINTER(_up), _up]),
    "sph_ns_neighbor_csr": (C.c_int, [_vp, C.c_uint, C.c_uint, C.POINTER(_up), C.POINTER(_up)]),
    "sph_dfsph_default_params": (None, [C.POINTER(DFSPHParams)]),
    "sph_dfsph_create": (C.c_int, [C.POINTER(DFSPHParams), C.POINTER(_vp)]),
    "sph_dfsph_destroy": (C.c_int, [_vp]),
    "sph_dfsph_set_fluid": (C.c_int, [_vp, _fp, _fp, C.c_size_t]),
    "sph_dfsph_reset": (C.c_int, [_vp]),
    "sph_dfsph_add_volume_map_mesh": (C.c_int, [_vp, _dp, C.c_size_t, _up, C.c_size_t, C.c_int, C.c_double, _up]),
    "sph_scene_load": (C.c_int, [C.c_char_p, C.POINTER(_vp)]),
    "sph_dfsph_write_particles": (C.c_int, [_vp, C.c_char_p, C.c_char_p]),
    "sph_dfsph_save_state": (C.c_int, [_vp, C.c_char_p]),
    "sph_dfsph_load_state": (C.c_int, [_vp, C.c_char_p]),
    "sph_bgeo_open": (C.c_int, [C.c_char_p, C.POINTER(_vp)]),
    "sph_bgeo_close": (C.c_int, [_vp]),
    "sph_bgeo_count": (C.c_int, [_vp, _szp, C.POINTER(C.c_int)]),
    "sph_bgeo_attribute": (C.c_int, [_vp, C.c_int, C.POINTER(C.c_char_p), C.POINTER(C.c_int), C.POINTER(C.c_int)]),
    "sph_bgeo_data": (C.c_int, [_vp, C.c_char_p, C.c_void_p, C.c_size_t]),
    "sph_bgeo_write": (C.c_int, [C.c_char_p, C.c_size_t, _fp, C.c_int, C.POINTER(C.c_char_p), C.POINTER(C.c_int),
                                 C.POINTER(C.c_int), C.POINTER(C.c_void_p)]),
    "sph_scene_destroy": (C.c_int, [_vp]),
    "sph_scene_params": (C.c_int, [_vp, C.c_void_p]),
    "sph_scene_counts": (C.c_int, [_vp, _szp, _szp, C.POINTER(C.c_int)]),
    "sph_scene_particles": (C.c_int, [_vp, _fp, _fp, _fp]),
    "sph_scene_body": (C.c_int, [_vp, C.c_int, C.POINTER(C.c_int), _dp, _dp, _dp, _dp, C.POINTER(C.c_int), _dp, _up]),
    "sph_scene_body_mesh": (C.c_int, [_vp, C.c_int, _dp, _szp, _up, _szp]),
    "sph_scene_emitter": (C.c_int, [_vp, C.c_int, C.c_void_p]),
    "sph_scene_emitter_settings": (C.c_int, [_vp, C.POINTER(C.c_int), _szp, C.POINTER(C.c_int), _dp, _dp]),
    "sph_scene_create_dfsph": (C.c_int, [_vp, C.POINTER(_vp)]),
    "sph_scene_simulation_method": (C.c_int, [_vp, C.POINTER(C.c_int), _dp, _dp]),
    "sph_dfsph_emit_particles": (C.c_int, [_vp, _fp, _fp, C.c_size_t]),
    "sph_dfsph_add_emitter": (C.c_int, [_vp, C.c_void_p]),
    "sph_dfsph_set_simulation_method": (C.c_int, [_vp, C.c_int]),
    "sph_dfsph_set_wcsph": (C.c_int, [_vp, C.c_double, C.c_double]),
    "sph_dfsph_set_emitter_reuse": (C.c_int, [_vp, C.c_int, _dp, _dp]),
    "sph_dfsph_set_max_emitter_particles": (C.c_int, [_vp, C.c_size_t]),
    "sph_dfsph_emitter_counts": (C.c_int, [_vp, _szp, _szp]),
    "sph_dfsph_add_boundary_particles": (C.c_int, [_vp, _fp, C.c_size_t]),
    "sph_dfsph_set_volume_map_box": (C.c_int, [_vp, _dp, _dp, C.c_int, C.c_double, _up]),
    "sph_dfsph_add_volume_map_sphere": (C.c_int, [_vp, _dp, C.c_double, C.c_int, C.c_double, _up]),
    "sph_dfsph_init": (C.c_int, [_vp]),
    "sph_dfsph_set_fluid_models": (C.c_int, [_vp, _up, C.c_size_t, _dp, C.c_uint]),
    "sph_dfsph_set_body_motion": (C.c_int, [_vp, C.c_uint, _dp, _dp, _dp, _dp, C.c_int]),
    "sph_dfsph_get_body_force": (C.c_int, [_vp, C.c_uint, _dp, _dp, C.c_int]),
    "sph_dfsph_get_body_reference": (C.c_int, [_vp, C.c_uint, _dp, _dp]),
    "sph_dfsph_set_batch_mode": (C.c_int, [C.c_int]),
    "sph_dfsph_batch_choice": (C.c_int, []),
    "sph_dfsph_step": (C.c_int, [_vp, C.c_int]),
    "sph_dfsph_step_batch": (C.c_int, [C.POINTER(_vp), C.c_size_t, C.c_int, C.c_int]),
    "sph_dfsph_stage": (C.c_int, [_vp, C.c_int]),
    "sph_dfsph_num_particles": (C.c_int, [_vp, _szp]),
    "sph_dfsph_get_field": (C.c_int, [_vp, C.c_char_p, _vp, C.c_size_t]),
    "sph_dfsph_set_field": (C.c_int, [_vp, C.c_char_p, _vp, C.c_size_t]),
    "sph_dfsph_get_neighbors": (C.c_int, [_vp, C.c_int, _up, _up, C.c_size_t, _szp]),
    "sph_dfsph_get_counters": (C.c_int, [_vp, C.POINTER(DFSPHCounters)]),
    "sph_dfsph_set_warm_start_model": (C.c_int, [_vp, C.c_int, _fp]),
    "sph_dfsph_collect_training": (C.c_int, [_vp, C.c_int, C.c_uint, C.c_size_t]),
    "sph_dfsph_set_warm_start_policy": (C.c_int, [_vp, C.c_int, C.c_int]),
    "sph_dfsph_set_warm_start_mode": (C.c_int, [_vp, C.c_int, C.c_int]),
    "sph_dfsph_get_training": (C.c_int, [_vp, C.c_int, _fp, _fp, C.c_size_t, _szp]),
    "sph_dfsph_set_time": (C.c_int, [_vp, C.c_double, C.c_double]),
    "sph_dfsph_enable_timing": (C.c_int, [_vp, C.c_int]),
    "sph_dfsph_time_only": (C.c_int, [_vp, C.c_char_p]),
    "sph_dfsph_set_lanes_per_particle": (C.c_int, [_vp, C.c_int]),
    "sph_dfsph_kernel_stats": (C.c_int, [_vp, C.c_int, C.POINTER(C.c_char_p), C.POINTER(C.c_longlong),
                                         _dp, C.POINTER(C.c_int)]),
    "sph_dfsph_reset_kernel_stats": (C.c_int, [_vp]),
    "sph_dfsph_synchronize": (C.c_int, [_vp]),
    "sph_kernel_eval": (C.c_int, [C.c_double, _fp, C.c_size_t, _fp, _fp]),
    "sph_mlp_num_params": (C.c_int, []),
    "sph_mlp_forward": (C.c_int, [_fp, _fp, C.c_size_t, _fp]),
    "sph_mlp_loss_grad": (C.c_int, [_fp, _fp, _fp, C.c_size_t, _fp, _fp]),
    "sph_mlp_train": (C.c_int, [_fp, _fp, _fp, C.c_size_t, C.c_int, C.c_int, C.c_double, C.c_uint, _fp]),
}


def lib():
    """Loads libsph_amd.so (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; "
                              f"g.build()'` (hipcc, gfx950)")
        L = C.CDLL(LIB_PATH)
        for name, (res, args) in _SIGS.items():
            f = getattr(L, name)
            f.restype = res
            f.argtypes = args
        _lib = L
    return _lib


def _chk(rc):
    if rc != 0:
        raise SPHError(rc, lib().sph_last_error().decode())


def device_count():
    n = C.c_int(0)
    _chk(lib().sph_device_count(C.byref(n)))
    return n.value


def synchronize():
    _chk(lib().sph_device_synchronize())


def kernel_eval(support_radius, r):
    """Device evaluation of the precomputed cubic kernel at FP32 offsets r."""
    r = np.ascontiguousarray(r, dtype=np.float32).reshape(-1, 3)
    n = len(r)
    w = np.zeros(n, np.float32)
    g = np.zeros((n, 3), np.float32)
    _chk(lib().sph_kernel_eval(support_radius, r.ctypes.data_as(_fp), n, w.ctypes.data_as(_fp),
                               g.ctypes.data_as(_fp)))
    return w, g


MLP_NPARAM = 4673


def _mlp_inputs(x):
    x = np.asarray(x, np.float32).reshape(len(x), -1)
    out = np.zeros((len(x), 8), np.float32)
    out[:, :min(6, x.shape[1])] = x[:, :6]
    return out


def mlp_forward(theta, x):
    """Device BF16-MFMA evaluation of the warm-start network on rows of 6
    features."""
    th = np.ascontiguousarray(theta, np.float32)
    xx = _mlp_inputs(x)
    y = np.zeros(len(xx), np.float32)
    _chk(lib().sph_mlp_forward(th.ctypes.data_as(_fp), xx.ctypes.data_as(_fp), len(xx), y.ctypes.data_as(_fp)))
    return y


def mlp_loss_grad(theta, x, t):
    th = np.ascontiguousarray(theta, np.float32)
    xx = _mlp_inputs(x)
    tt = np.ascontiguousarray(t, np.float32)
    g = np.zeros(MLP_NPARAM, np.float32)
    loss = C.c_float(0)
    _chk(lib().sph_mlp_loss_grad(th.ctypes.data_as(_fp), xx.ctypes.data_as(_fp), tt.ctypes.data_as(_fp), len(xx),
                                 g.ctypes.data_as(_fp), C.byref(loss)))
    return loss.value, g


def mlp_train(theta, x, t, steps=1000, batch=4096, lr=1e-3, seed=0):
    """Adam on the device; returns (new theta, final loss)."""
    th = np.ascontiguousarray(theta, np.float32).copy()
    xx = _mlp_inputs(x)
    tt = np.ascontiguousarray(t, np.float32)
    loss = C.c_float(0)
    _chk(lib().sph_mlp_train(th.ctypes.data_as(_fp), xx.ctypes.data_as(_fp), tt.ctypes.data_as(_fp), len(xx),
                             steps, batch, lr, seed, C.byref(loss)))
    return th, loss.value


def step_batch(sims, n_steps=1, threads=0):
    """Steps the TimeStepDFSPH handles `sims` together (sph_dfsph_step_batch)."""
    arr = (_vp * len(sims))(*[s.h for s in sims])
    _chk(lib().sph_dfsph_step_batch(arr, len(sims), int(n_steps), int(threads)))
    for s in sims:
        s._refresh_n()


BATCH_MODES = {"threads": 0, "batched": 1, "graphs": 2, "auto": 3}


def set_batch_mode(mode):
    """How step_batch runs: "threads" (scene by scene on host threads),
    "batched" (the solves of all scenes in batched launches), "graphs"
    (batched, replayed from captured HIP graphs) or "auto" (the default: the
    faster of "threads" and "graphs", timed on the first steps of each set of
    handles)."""
    _chk(lib().sph_dfsph_set_batch_mode(BATCH_MODES[mode] if isinstance(mode, str) else int(mode)))


def batch_choice():
    """The way "auto" chose for the last set of handles ("threads" or
    "graphs"), or None while it is still timing."""
    c = lib().sph_dfsph_batch_choice()
    return {0: "threads", 2: "graphs"}.get(c)


class PointSet:
    """View of one point set (CompactNSearch::PointSet)."""

    def __init__(self, ns, index):
        self._ns = ns
        self.index = index

    def n_points(self):
        n = C.c_size_t(0)
        _chk(lib().sph_ns_n_points(self._ns.h, self.index, C.byref(n)))
        return n.value

    def n_neighbors(self, set_j, i):
        out = C.c_uint(0)
        _chk(lib().sph_ns_n_neighbors(self._ns.h, self.index, set_j, i, C.byref(out)))
        return out.value

    def neighbor(self, set_j, i, k):
        out = C.c_uint(0)
        _chk(lib().sph_ns_neighbor(self._ns.h, self.index, set_j, i, k, C.byref(out)))
        return out.value

    def neighbor_list(self, set_j, i):
        p = _up()
        cnt = C.c_uint(0)
        _chk(lib().sph_ns_neighbor_list(self._ns.h, self.index, set_j, i, C.byref(p), C.byref(cnt)))
        return np.ctypeslib.as_array(p, shape=(cnt.value,)).copy() if cnt.value else np.zeros(0, np.uint32)

    def sort_field(self, arr):
        """Permutes arr (first axis = points) in place with the last z_sort."""
        assert arr.flags.c_contiguous
        _chk(lib().sph_ns_sort_field(self._ns.h, self.index, arr.ctypes.data, arr.nbytes // max(len(arr), 1)))

    def get_user_data(self):
        out = _vp()
        _chk(lib().sph_ns_user_data(self._ns.h, self.index, C.byref(out)))
        return out.value


class NeighborhoodSearch:
    """Drop-in for CompactNSearch::NeighborhoodSearch on the device."""

    def __init__(self, radius, erase_empty_cells=False):
        h = _vp()
        _chk(lib().sph_ns_create(radius, int(erase_empty_cells), C.byref(h)))
        self.h = h
        self._arrays = []

    def __del__(self):
        if getattr(self, "h", None) and _lib is not None:
            _lib.sph_ns_destroy(self.h)
            self.h = None

    def set_radius(self, r):
        _chk(lib().sph_ns_set_radius(self.h, r))

    def radius(self):
        r = C.c_double(0)
        _chk(lib().sph_ns_get_radius(self.h, C.byref(r)))
        return r.value

    def reset(self):
        _chk(lib().sph_ns_reset(self.h))
        self._arrays = []

    def add_point_set(self, x, is_dynamic=True, search_neighbors=True, find_neighbors=True):
        """x: C-contiguous (n, 3) float32 or float64 array, kept by reference
        (the library reads it on update_point_sets/find_neighbors)."""
        assert x.flags.c_contiguous and x.ndim == 2 and x.shape[1] == 3
        dtype = SPH_F64 if x.dtype == np.float64 else SPH_F32
        assert x.dtype in (np.float32, np.float64)
        idx = C.c_uint(0)
        _chk(lib().sph_ns_add_point_set(self.h, x.ctypes.data, len(x), dtype, int(is_dynamic),
                                        int(search_neighbors), int(find_neighbors), None, C.byref(idx)))
        self._arrays.append(x)
        return idx.value

    def resize_point_set(self, i, x):
        assert x.flags.c_contiguous
        _chk(lib().sph_ns_resize_point_set(self.h, i, x.ctypes.data, len(x)))
        self._arrays[i] = x

    def update_point_sets(self):
        _chk(lib().sph_ns_update_point_sets(self.h))

    def find_neighbors(self, points_changed=True):
        _chk(lib().sph_ns_find_neighbors(self.h, int(points_changed)))

    def find_neighbors_point(self, x, set_j, cap=4096):
        out = np.zeros(cap, np.uint32)
        cnt = C.c_uint(0)
        xx = np.ascontiguousarray(x, np.float64)
        _chk(lib().sph_ns_query_point(self.h, xx.ctypes.data_as(_dp), set_j, out.ctypes.data_as(_up), cap,
                                      C.byref(cnt)))
        return out[: min(cnt.value, cap)]

    def z_sort(self):
        _chk(lib().sph_ns_z_sort(self.h))

    def set_active(self, *args):
        if len(args) == 1:
            _chk(lib().sph_ns_set_active_all(self.h, int(args[0])))
        elif len(args) == 3 and isinstance(args[2], bool) and isinstance(args[1], int) and not isinstance(args[1], bool):
            _chk(lib().sph_ns_set_active_pair(self.h, args[0], args[1], int(args[2])))
        else:
            i, s, f = args[0], args[1] if len(args) > 1 else True, args[2] if len(args) > 2 else True
            _chk(lib().sph_ns_set_active_set(self.h, i, int(s), int(f)))

    def is_active(self, i, j):
        out = C.c_int(0)
        _chk(lib().sph_ns_is_active_pair(self.h, i, j, C.byref(out)))
        return bool(out.value)

    def n_point_sets(self):
        out = C.c_uint(0)
        _chk(lib().sph_ns_n_point_sets(self.h, C.byref(out)))
        return out.value

    def point_set(self, i):
        return PointSet(self, i)

    def neighbors_csr(self, i, j):
        """(offsets, indices) copies of all lists of set i in set j."""
        po, pi = _up(), _up()
        _chk(lib().sph_ns_neighbor_csr(self.h, i, j, C.byref(po), C.byref(pi)))
        n = self.point_set(i).n_points()
        off = np.ctypeslib.as_array(po, shape=(n + 1,)).copy()
        idx = np.ctypeslib.as_array(pi, shape=(int(off[-1]),)).copy() if off[-1] else np.zeros(0, np.uint32)
        return off, idx


class Scene:
    """A SPlisHSPlasH scene file read by the library (sph_scene_load):
    parameters, sampled fluid blocks, static bodies and emitters."""

    def __init__(self, path):
        h = _vp()
        _chk(lib().sph_scene_load(os.fsencode(path), C.byref(h)))
        self.h = h
        self.params = DFSPHParams()
        _chk(lib().sph_scene_params(self.h, C.byref(self.params)))
        nf, nb, nbod = C.c_size_t(), C.c_size_t(), C.c_int()
        _chk(lib().sph_scene_counts(self.h, C.byref(nf), C.byref(nb), C.byref(nbod)))
        self.n, self.nb, self.nbodies = nf.value, nb.value, nbod.value

    def __del__(self):
        if getattr(self, "h", None) and _lib is not None:
            _lib.sph_scene_destroy(self.h)
            self.h = None

    def particles(self):
        """(x, v, boundary_x) as float32 arrays of shape (n, 3)."""
        x = np.zeros((self.n, 3), np.float32)
        v = np.zeros((self.n, 3), np.float32)
        bx = np.zeros((self.nb, 3), np.float32)
        _chk(lib().sph_scene_particles(self.h, x.ctypes.data_as(_fp), v.ctypes.data_as(_fp), bx.ctypes.data_as(_fp)))
        return x, v, bx

    def body(self, k):
        kind, inv = C.c_int(), C.c_int()
        lo, hi, cen = (np.zeros(3) for _ in range(3))
        rad, th = C.c_double(), C.c_double()
        res = np.zeros(3, np.uint32)
        _chk(lib().sph_scene_body(self.h, k, C.byref(kind), lo.ctypes.data_as(_dp), hi.ctypes.data_as(_dp),
                                  cen.ctypes.data_as(_dp), C.byref(rad), C.byref(inv), C.byref(th),
                                  res.ctypes.data_as(_up)))
        return {"kind": ("box", "sphere", "mesh")[kind.value], "lo": lo, "hi": hi, "centre": cen,
                "radius": rad.value, "invert": bool(inv.value), "thickness": th.value, "resolution": res}

    def body_mesh(self, k):
        """(vertices (m, 3), faces (f, 3)) of mesh body k, world coordinates."""
        nv, nf = C.c_size_t(), C.c_size_t()
        _chk(lib().sph_scene_body_mesh(self.h, k, None, C.byref(nv), None, C.byref(nf)))
        v = np.zeros((nv.value, 3))
        f = np.zeros((nf.value, 3), np.uint32)
        _chk(lib().sph_scene_body_mesh(self.h, k, v.ctypes.data_as(_dp), C.byref(nv), f.ctypes.data_as(_up),
                                       C.byref(nf)))
        return v, f

    def emitters(self):
        """The scene's emitters as dicts, and the fluid's emitter settings."""
        n, me, ru = C.c_int(), C.c_size_t(), C.c_int()
        lo, hi = np.zeros(3), np.zeros(3)
        _chk(lib().sph_scene_emitter_settings(self.h, C.byref(n), C.byref(me), C.byref(ru), lo.ctypes.data_as(_dp),
                                              hi.ctypes.data_as(_dp)))
        out = []
        for k in range(n.value):
            e = Emitter()
            _chk(lib().sph_scene_emitter(self.h, k, C.byref(e)))
            out.append({"type": e.type, "width": e.width, "height": e.height, "translation": np.array(e.translation[:]),
                        "rotation": np.array(e.rotation[:]).reshape(3, 3), "velocity": e.velocity,
                        "emit_start_time": e.emit_start_time, "emit_end_time": e.emit_end_time})
        return out, {"max_emitter_particles": me.value, "reuse": bool(ru.value), "box_min": lo, "box_max": hi}

    def simulation_method(self):
        """The scene's simulationMethod and, for WCSPH, its stiffness and
        exponent: (method, stiffness, exponent)."""
        m, k, g = C.c_int(), C.c_double(), C.c_double()
        _chk(lib().sph_scene_simulation_method(self.h, C.byref(m), C.byref(k), C.byref(g)))
        return m.value, k.value, g.value

    def create_dfsph(self):
        """A TimeStepDFSPH with the scene's parameters, fluid and boundaries."""
        h = _vp()
        _chk(lib().sph_scene_create_dfsph(self.h, C.byref(h)))
        return TimeStepDFSPH(self.params, _handle=h, _n=self.n, _nb=self.nb)


def read_bgeo(path):
    """A partio BGEO file as {"position": (n, 3) float32, attribute name:
    array} (float attributes float32, int attributes int32, vectors (n, k))."""
    h = _vp()
    _chk(lib().sph_bgeo_open(os.fsencode(path), C.byref(h)))
    try:
        n, na = C.c_size_t(), C.c_int()
        _chk(lib().sph_bgeo_count(h, C.byref(n), C.byref(na)))
        out = {}
        pos = np.zeros((n.value, 3), np.float32)
        _chk(lib().sph_bgeo_data(h, b"position", pos.ctypes.data_as(C.c_void_p), pos.nbytes))
        out["position"] = pos
        for k in range(na.value):
            nm, ty, sz = C.c_char_p(), C.c_int(), C.c_int()
            _chk(lib().sph_bgeo_attribute(h, k, C.byref(nm), C.byref(ty), C.byref(sz)))
            a = np.zeros((n.value, sz.value), np.int32 if ty.value == 1 else np.float32)
            _chk(lib().sph_bgeo_data(h, nm.value, a.ctypes.data_as(C.c_void_p), a.nbytes))
            out[nm.value.decode()] = a[:, 0] if sz.value == 1 else a
        return out
    finally:
        lib().sph_bgeo_close(h)


def write_bgeo(path, position, attrs):
    """Writes a BGEO file: `attrs` maps names to (n,) or (n, k) arrays; int
    arrays become int attributes, (n, 3) float arrays vectors."""
    pos = np.ascontiguousarray(position, np.float32).reshape(-1, 3)
    names, types, sizes, bufs = [], [], [], []
    for nm, a in attrs.items():
        a = np.asarray(a)
        isint = np.issubdtype(a.dtype, np.integer)
        a = np.ascontiguousarray(a, np.int32 if isint else np.float32).reshape(len(pos), a.shape[1] if a.ndim == 2 else 1)
        names.append(nm.encode())
        types.append(1 if isint else (5 if a.shape[1] == 3 else 0))
        sizes.append(a.shape[1])
        bufs.append(a)
    k = len(names)
    cn = (C.c_char_p * max(k, 1))(*names)
    ct = (C.c_int * max(k, 1))(*types)
    cs = (C.c_int * max(k, 1))(*sizes)
    cd = (C.c_void_p * max(k, 1))(*[b.ctypes.data for b in bufs])
    _chk(lib().sph_bgeo_write(os.fsencode(path), len(pos), pos.ctypes.data_as(_fp), k, cn, ct, cs, cd))


def load_scene(path):
    """Reads a scene file and returns a ready-to-step TimeStepDFSPH."""
    return Scene(path).create_dfsph()


class TimeStepDFSPH:
    """Device-resident DFSPH time step (SPH::TimeStepDFSPH) with the fluid,
    Akinci2012 boundary particles or a Bender2019 volume-map box."""

    def __init__(self, params=None, _handle=None, _n=0, _nb=0, **kw):
        self.params = params if params is not None else default_params(**kw)
        if _handle is None:
            h = _vp()
            _chk(lib().sph_dfsph_create(C.byref(self.params), C.byref(h)))
        else:
            h = _handle
        self.h = h
        self.n = _n
        self.nb = _nb

    def __del__(self):
        if getattr(self, "h", None) and _lib is not None:
            _lib.sph_dfsph_destroy(self.h)
            self.h = None

    def set_fluid(self, x, v=None):
        x = np.ascontiguousarray(x, dtype=np.float32).reshape(-1, 3)
        v = np.zeros_like(x) if v is None else np.ascontiguousarray(v, dtype=np.float32).reshape(-1, 3)
        self.n = len(x)
        _chk(lib().sph_dfsph_set_fluid(self.h, x.ctypes.data_as(_fp), v.ctypes.data_as(_fp), self.n))

    def add_boundary_particles(self, x):
        x = np.ascontiguousarray(x, dtype=np.float32).reshape(-1, 3)
        self.nb += len(x)
        _chk(lib().sph_dfsph_add_boundary_particles(self.h, x.ctypes.data_as(_fp), len(x)))

    def set_volume_map_box(self, lo, hi, res, invert=True, thickness=0.0):
        lo = np.ascontiguousarray(lo, np.float64)
        hi = np.ascontiguousarray(hi, np.float64)
        r = np.ascontiguousarray(res, np.uint32)
        _chk(lib().sph_dfsph_set_volume_map_box(self.h, lo.ctypes.data_as(_dp), hi.ctypes.data_as(_dp),
                                                int(invert), thickness, r.ctypes.data_as(_up)))

    def add_volume_map_sphere(self, centre, radius, res, invert=False, thickness=0.0):
        """Static sphere obstacle as a Bender2019 volume map; `res` is the
        cells per axis or, as a float, the cell size in metres."""
        c = np.ascontiguousarray(centre, np.float64)
        if np.ndim(res) == 0:
            ext = 2.0 * (radius + 8.0 * 4.0 * self.params.particle_radius + thickness)
            res = [max(1, int(round(ext / float(res))))] * 3
        r = np.ascontiguousarray(res, np.uint32)
        _chk(lib().sph_dfsph_add_volume_map_sphere(self.h, c.ctypes.data_as(_dp), float(radius), int(invert),
                                                   thickness, r.ctypes.data_as(_up)))

    def add_volume_map_mesh(self, vertices, faces, res, invert=False, thickness=0.0):
        """Static closed triangle mesh (world coordinates) as a Bender2019
        volume map with res[0..2] cells over its box grown by 8h."""
        v = np.ascontiguousarray(vertices, np.float64).reshape(-1, 3)
        f = np.ascontiguousarray(faces, np.uint32).reshape(-1, 3)
        r = np.ascontiguousarray(res, np.uint32)
        _chk(lib().sph_dfsph_add_volume_map_mesh(self.h, v.ctypes.data_as(_dp), len(v), f.ctypes.data_as(_up), len(f),
                                                 int(invert), thickness, r.ctypes.data_as(_up)))

    def init(self):
        _chk(lib().sph_dfsph_init(self.h))

    def reset(self):
        """TimeStepDFSPH::reset: solver fields and iteration counters to zero."""
        _chk(lib().sph_dfsph_reset(self.h))

    def write_particles(self, path, fields="velocity"):
        """The exporter's BGEO particle file (position, id and `fields`,
        ';'-separated)."""
        _chk(lib().sph_dfsph_write_particles(self.h, os.fsencode(path), fields.encode()))

    def save_state(self, prefix):
        _chk(lib().sph_dfsph_save_state(self.h, os.fsencode(prefix)))

    def load_state(self, prefix):
        """Sets every field the state file holds and the time; the handle
        grows to the file's particle count."""
        _chk(lib().sph_dfsph_load_state(self.h, os.fsencode(prefix)))
        self._refresh_n()

    def emit_particles(self, x, v=None):
        """Appends particles (emitter + emittedParticles): ids continue from
        the current count, stiffness starts at zero."""
        x = np.ascontiguousarray(x, dtype=np.float32).reshape(-1, 3)
        v = np.zeros_like(x) if v is None else np.ascontiguousarray(v, dtype=np.float32).reshape(-1, 3)
        _chk(lib().sph_dfsph_emit_particles(self.h, x.ctypes.data_as(_fp), v.ctypes.data_as(_fp), len(x)))
        self.n += len(x)

    def set_simulation_method(self, method):
        """Simulation::setSimulationMethod for this handle: METHOD_DFSPH (4),
        METHOD_PCISPH (1), METHOD_IISPH (3) or METHOD_WCSPH (0)."""
        _chk(lib().sph_dfsph_set_simulation_method(self.h, int(method)))

    def set_wcsph(self, stiffness=50.0, exponent=7.0):
        """TimeStepWCSPH's stiffness and exponent of the state equation
        p = stiffness ((rho / rho0)^exponent - 1) (TimeStepWCSPH.cpp:56-63,
        106); both at least 1e-6."""
        _chk(lib().sph_dfsph_set_wcsph(self.h, float(stiffness), float(exponent)))

    def add_emitter(self, width, height, pos, rotation, velocity, type=0, emit_start_time=0.0,
                    emit_end_time=float(np.finfo(np.float64).max)):
        """EmitterSystem::addEmitter (EmitterSystem.cpp:93-104) with the
        emitter's start and end times; `rotation` is a 3x3 matrix whose
        column 0 is the emit direction."""
        e = Emitter()
        e.type = int(type)
        e.width = int(width)
        e.height = int(height)
        e.translation[:] = [float(c) for c in np.asarray(pos, np.float64).ravel()[:3]]
        e.rotation[:] = [float(c) for c in np.asarray(rotation, np.float64).reshape(9)]
        e.velocity = float(velocity)
        e.emit_start_time = float(emit_start_time)
        e.emit_end_time = float(emit_end_time)
        _chk(lib().sph_dfsph_add_emitter(self.h, C.byref(e)))

    def enable_reuse_particles(self, box_min=(-1.0, -1.0, -1.0), box_max=(1.0, 1.0, 1.0)):
        """EmitterSystem::enableReuseParticles (EmitterSystem.cpp:106-111)."""
        lo = np.ascontiguousarray(box_min, np.float64)
        hi = np.ascontiguousarray(box_max, np.float64)
        _chk(lib().sph_dfsph_set_emitter_reuse(self.h, 1, lo.ctypes.data_as(_dp), hi.ctypes.data_as(_dp)))

    def disable_reuse_particles(self):
        _chk(lib().sph_dfsph_set_emitter_reuse(self.h, 0, None, None))

    def set_max_emitter_particles(self, m):
        _chk(lib().sph_dfsph_set_max_emitter_particles(self.h, int(m)))

    def set_fluid_models(self, model, materials):
        """Several fluid models: `model` gives each particle's model (caller
        order), each material a dict with density0 and optionally viscosity,
        viscosity_boundary, xsph, xsph_boundary (default: the parameters')."""
        m = np.ascontiguousarray(model, np.uint32)
        p = self.params
        mat = np.ascontiguousarray([[d["density0"], d.get("viscosity", p.viscosity),
                                     d.get("viscosity_boundary", p.viscosity_boundary), d.get("xsph", p.xsph),
                                     d.get("xsph_boundary", p.xsph_boundary)] for d in materials], np.float64)
        _chk(lib().sph_dfsph_set_fluid_models(self.h, m.ctypes.data_as(_up), len(m), mat.ctypes.data_as(_dp),
                                              len(materials)))

    def set_body_motion(self, obj, position, rotation=None, velocity=(0.0, 0.0, 0.0),
                        angular_velocity=(0.0, 0.0, 0.0), kind="dynamic"):
        """RigidBodyObject state of boundary object `obj` (volume maps in
        insertion order): position of its reference point, 3x3 rotation,
        velocity, angular velocity; kind "static", "animated" or "dynamic"."""
        R = np.eye(3) if rotation is None else np.asarray(rotation, np.float64).reshape(3, 3)
        k = {"static": 0, "animated": 1, "dynamic": 2}[kind]
        d = lambda a: np.ascontiguousarray(a, np.float64).ravel()
        p, Rr, v, w = d(position), d(R), d(velocity), d(angular_velocity)
        _chk(lib().sph_dfsph_set_body_motion(self.h, int(obj), p.ctypes.data_as(_dp), Rr.ctypes.data_as(_dp),
                                             v.ctypes.data_as(_dp), w.ctypes.data_as(_dp), k))

    def body_force(self, obj, clear=True):
        """(force, torque) the fluid exerted on dynamic body `obj` since the last clear."""
        f, t = np.zeros(3), np.zeros(3)
        _chk(lib().sph_dfsph_get_body_force(self.h, int(obj), f.ctypes.data_as(_dp), t.ctypes.data_as(_dp),
                                            int(clear)))
        return f, t

    def body_reference(self, obj):
        """(reference point where the shape was given, largest vertex distance from it)."""
        p, m = np.zeros(3), np.zeros(1)
        _chk(lib().sph_dfsph_get_body_reference(self.h, int(obj), p.ctypes.data_as(_dp), m.ctypes.data_as(_dp)))
        return p, float(m[0])

    def emitter_counts(self):
        """(sum of emitted particles, sum of reused particles)."""
        e, r = C.c_size_t(0), C.c_size_t(0)
        _chk(lib().sph_dfsph_emitter_counts(self.h, C.byref(e), C.byref(r)))
        return e.value, r.value

    def _refresh_n(self):
        n = C.c_size_t(0)
        _chk(lib().sph_dfsph_num_particles(self.h, C.byref(n)))
        self.n = n.value

    def step(self, n=1):
        _chk(lib().sph_dfsph_step(self.h, n))
        self._refresh_n()

    def stage(self, name):
        _chk(lib().sph_dfsph_stage(self.h, STAGES[name] if isinstance(name, str) else int(name)))
        self._refresh_n()

    def get(self, name):
        if name == "boundary particle volume":
            out = np.zeros(self.nb, np.float32)
        else:
            if (name.startswith("boundary x ") or name.startswith("boundary volume ") or
                    name.startswith("boundary density")):
                # per map object; density maps: "boundary density [o]" and
                # "boundary density gradient [o]"
                comps = 3 if (name.startswith("boundary x") or name.startswith("boundary density gradient")) else 1
            else:
                comps = FIELD_COMPONENTS[name]
            dt = np.uint32 if name in ("id", "state", "fluid model", "fluid neighbor count",
                                       "boundary neighbor count") else np.float32
            out = np.zeros((self.n, comps) if comps > 1 else self.n, dt)
        _chk(lib().sph_dfsph_get_field(self.h, name.encode(), out.ctypes.data, out.nbytes))
        return out

    def set(self, name, values):
        a = np.ascontiguousarray(values, dtype=np.uint32 if name == "state" else np.float32)
        _chk(lib().sph_dfsph_set_field(self.h, name.encode(), a.ctypes.data, a.nbytes))

    def neighbors(self, boundary=False):
        off = np.zeros(self.n + 1, np.uint32)
        nnz = C.c_size_t(0)
        _chk(lib().sph_dfsph_get_neighbors(self.h, int(boundary), off.ctypes.data_as(_up), None, 0, C.byref(nnz)))
        idx = np.zeros(max(nnz.value, 1), np.uint32)
        _chk(lib().sph_dfsph_get_neighbors(self.h, int(boundary), off.ctypes.data_as(_up),
                                           idx.ctypes.data_as(_up), idx.size, C.byref(nnz)))
        return off, idx[: nnz.value]

    def counters(self):
        c = DFSPHCounters()
        _chk(lib().sph_dfsph_get_counters(self.h, C.byref(c)))
        return c.as_dict()

    def set_time(self, t, dt):
        _chk(lib().sph_dfsph_set_time(self.h, t, dt))

    _SOLVERS = {"pressure": 0, "divergence": 1}

    def set_warm_start_model(self, solver, theta):
        """Start `solver` ("pressure" or "divergence") from the network with
        parameters `theta` (per particle, where its initial residual beats
        the reference's warm start); None restores the reference's start."""
        s = self._SOLVERS[solver]
        if theta is None:
            _chk(lib().sph_dfsph_set_warm_start_model(self.h, s, None))
            return
        th = np.ascontiguousarray(theta, np.float32)
        if th.size != MLP_NPARAM:
            raise ValueError(f"theta must hold {MLP_NPARAM} floats")
        self._theta = getattr(self, "_theta", {})
        self._theta[solver] = th
        _chk(lib().sph_dfsph_set_warm_start_model(self.h, s, th.ctypes.data_as(_fp)))

    WARM_START_MODES = {"reference": 0, "previous": 1, "network": 2}

    def set_warm_start_mode(self, solver, mode):
        """Start of `solver`'s solves: "reference" (0), "previous" (1, the
        previous step's full stiffness) or "network" (2)."""
        m = self.WARM_START_MODES[mode] if isinstance(mode, str) else int(mode)
        _chk(lib().sph_dfsph_set_warm_start_mode(self.h, self._SOLVERS[solver], m))

    def set_warm_start_policy(self, solver, min_prev_iterations):
        """Use the network for `solver` only when its previous solve took at
        least this many iterations (0: always)."""
        _chk(lib().sph_dfsph_set_warm_start_policy(self.h, self._SOLVERS[solver], int(min_prev_iterations)))

    def collect_training(self, solver, stride, capacity):
        """Records (features, converged stiffness / scale) of every
        `stride`-th particle after each solve, up to `capacity` samples;
        stride 0 stops recording."""
        self._cap = getattr(self, "_cap", {})
        self._cap[solver] = int(capacity)
        _chk(lib().sph_dfsph_collect_training(self.h, self._SOLVERS[solver], int(stride), int(capacity)))

    def get_training(self, solver):
        """Returns (x [k, 8], t [k]) recorded since the last call and clears
        the record."""
        cap = getattr(self, "_cap", {}).get(solver, 0)
        x = np.zeros((max(cap, 1), 8), np.float32)
        t = np.zeros(max(cap, 1), np.float32)
        n = C.c_size_t(0)
        _chk(lib().sph_dfsph_get_training(self.h, self._SOLVERS[solver], x.ctypes.data_as(_fp),
                                          t.ctypes.data_as(_fp), cap, C.byref(n)))
        return x[: n.value].copy(), t[: n.value].copy()

    def enable_timing(self, on=True):
        _chk(lib().sph_dfsph_enable_timing(self.h, int(on)))

    def set_lanes_per_particle(self, lanes):
        """1, 2 or 4 lanes per particle in the solver sweeps; 0: by rule."""
        _chk(lib().sph_dfsph_set_lanes_per_particle(self.h, int(lanes)))

    def time_only(self, names):
        """Restrict timing to these kernel names (None: all)."""
        _chk(lib().sph_dfsph_time_only(self.h, ",".join(names).encode() if names else None))

    def reset_kernel_stats(self):
        _chk(lib().sph_dfsph_reset_kernel_stats(self.h))

    def kernel_stats(self):
        cnt = C.c_int(0)
        _chk(lib().sph_dfsph_kernel_stats(self.h, -1, None, None, None, C.byref(cnt)))
        out = {}
        for k in range(cnt.value):
            nm = C.c_char_p()
            la = C.c_longlong(0)
            ms = C.c_double(0)
            _chk(lib().sph_dfsph_kernel_stats(self.h, k, C.byref(nm), C.byref(la), C.byref(ms), C.byref(cnt)))
            out[nm.value.decode()] = (la.value, ms.value)
        return out

    def synchronize(self):
        _chk(lib().sph_dfsph_synchronize(self.h))
