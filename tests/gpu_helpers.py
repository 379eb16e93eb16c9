"""Shared helpers of the GPU parity tests: seeded inputs, host<->device
conversion and error norms."""

import ctypes
import sys

import numpy as np
import torch


def say(*a):
    """Print and flush what names the case before each GPU step."""
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def host(t):
    return t.detach().cpu().numpy()


def rel_l2(got, want, floor=0.0):
    got, want = np.asarray(got), np.asarray(want)
    den = max(np.linalg.norm(want), floor)
    if den == 0:
        return float(np.linalg.norm(got))
    return float(np.linalg.norm(got - want) / den)


def smooth_field(rng, n, amp=1.0, zero_rim=1):
    """A smooth random (n, n) field with a zero rim of zero_rim cells."""
    a = rng.standard_normal((n, n))
    k = np.array([.25, .5, .25])
    for _ in range(4):
        a = (np.roll(a, 1, 0) + 2 * a + np.roll(a, -1, 0)) / 4
        a = (np.roll(a, 1, 1) + 2 * a + np.roll(a, -1, 1)) / 4
    del k
    if zero_rim:
        a[:zero_rim] = a[-zero_rim:] = 0
        a[:, :zero_rim] = a[:, -zero_rim:] = 0
    return amp * a / np.abs(a).max()


def perturbed_state(oracle, cfg, seed=0, amp_x=None, amp_p=.05, amp_f=.05):
    """init() plus smooth offsets, momenta, fields and densities: a
    non-trivial `prev` for one-step comparisons."""
    xs, ys, const, vp, st = oracle.init(cfg)
    rng = np.random.default_rng(seed)
    nc = const.m.shape[0]
    n = cfg.grid_steps
    h = cfg.grid_step_size
    amp_x = 2 * h if amp_x is None else amp_x
    for name in ("x_offt", "y_offt"):
        setattr(st, name, smooth_field(rng, nc, amp_x, zero_rim=0))
    for name in ("px", "py", "pz"):
        setattr(st, name, smooth_field(rng, nc, amp_p, zero_rim=0))
    for name in ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "jx", "jy", "jz"):
        setattr(st, name, smooth_field(rng, n, amp_f, zero_rim=2))
    st.ro = smooth_field(rng, n, amp_f, zero_rim=2)
    return xs, ys, const, vp, st


def to_device_state(lc, st):
    return lc.GPUArrays(**{k: dev(getattr(st, k)) for k in (
        "x_offt", "y_offt", "px", "py", "pz", "Ex", "Ey", "Ez", "Bx", "By",
        "Bz", "ro", "jx", "jy", "jz")})


STATE = ("x_offt", "y_offt", "px", "py", "pz", "Ex", "Ey", "Ez", "Bx", "By",
         "Bz", "ro", "jx", "jy", "jz")


class Workspace:
    """One workspace of the C ABI, apart from those the package keeps, with the
    plasma of oracle.init(cfg), and operators on it."""

    def __init__(self, oracle, cfg):
        from lcode3d_amd import _lib
        from lcode3d_amd import lcode as L
        self.lib, self.cfg = _lib.load(), cfg
        _, _, self.const, self.vp, _ = oracle.init(cfg)
        self.shape = self.const.m.shape
        self.keep = [dev(getattr(self.vp, k)) for k in (
            "influence_prev", "influence_next", "fine_grid", "indices_prev", "indices_next")]
        self.cvp = _lib.LcodeVirtParams(*(t.data_ptr() for t in self.keep))
        self.cs = L._config_struct(cfg, self.shape[0], self.keep[2].numel())
        self.ws = ctypes.c_void_p()
        _lib.check(self.lib.lcode_workspace_create(ctypes.byref(self.cs), ctypes.byref(self.ws)),
                   "create")
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.m, self.q, self.x, self.y, self.ro0 = (
            dev(getattr(self.const, k)) for k in ("m", "q", "x_init", "y_init", "ro_initial"))

    def push(self, xo, yo, p):
        n = self.cfg.grid_steps
        fields = [torch.zeros((n, n), dtype=torch.float64, device="cuda") for _ in range(6)]
        ins = [self.m, self.q, self.x, self.y, xo, yo, xo, yo, *p]
        outs = [torch.empty_like(xo) for _ in range(5)]
        ptrs = lambda ts: (ctypes.c_void_p * len(ts))(*(t.data_ptr() for t in ts))  # noqa: E731
        rc = self.lib.lcode_move_smart(self.ws, ctypes.byref(self.cs),
                                       *[t.data_ptr() for t in ins], ptrs(fields), ptrs(outs),
                                       self.stream)
        torch.cuda.synchronize()
        assert rc == 0, self.lib.lcode_last_error()
        return outs

    def deposit(self, xo, yo, p, noalloc=False):
        n = self.cfg.grid_steps
        outs = [torch.empty((n, n), dtype=torch.float64, device="cuda") for _ in range(4)]
        parts = [xo, yo, self.m, self.q, *p]
        args = (ctypes.byref(self.cs), self.ro0.data_ptr(), *[t.data_ptr() for t in parts],
                ctypes.byref(self.cvp), (ctypes.c_void_p * 4)(*(o.data_ptr() for o in outs)),
                self.stream)
        rc = (self.lib.lcode_deposit_noalloc(*args) if noalloc
              else self.lib.lcode_deposit(self.ws, *args))
        torch.cuda.synchronize()
        assert rc == 0, self.lib.lcode_last_error()
        return outs

    def nonfinite(self):
        flag = ctypes.c_int32()
        self.lib.lcode_workspace_nonfinite(self.ws, 0, ctypes.byref(flag))
        return flag.value

    def faults(self):
        count = ctypes.c_int64()
        self.lib.lcode_workspace_fault_count(self.ws, self.stream, ctypes.byref(count))
        return count.value

    def close(self):
        torch.cuda.synchronize()
        self.lib.lcode_workspace_destroy(self.ws)
