"""The FP64 LU and substitutions of the workgroup kernels (csrc/kernels/odemi_lu.h)
alone, against the element-by-element LU of the CPU restatement, bit for bit: odd
and even n at the edges of panels (8 columns), tiles (16) and row slots (64), four
and eight waves, row strides of n and more, and the matrices that the rules of
the pivot search and of the short quotients are for."""
import ctypes
import os

import numpy as np
import pytest

import oracle as O
from odemi import _lib

SIZES = {64: (1, 2, 3, 5, 7, 8, 9, 15, 16, 17, 24, 31, 33, 48, 63, 64),
         128: (65, 66, 71, 72, 73, 79, 81, 96, 97, 111, 120, 127, 128),
         135: (7, 64, 65, 128, 129, 130, 131, 133, 135)}
MAX_LDS = 160 * 1024


def lds_bytes(n, ld):
    return ((n * ld + n) * 8 + 15) // 16 * 16 + 64 + 4 * n


def matrices(n):
    """(name, A, b) for one n; the same on every run."""
    r = np.random.default_rng(n)
    g = lambda *s: r.normal(size=s)
    out = [("normal", g(n, n), g(n))]
    band = np.where(abs(np.subtract.outer(np.arange(n), np.arange(n))) <= 1, g(n, n), 0.0) - 4 * np.eye(n)
    out.append(("band", band, g(n)))
    out.append(("ties", r.choice([-1.0, 1.0], (n, n)), g(n)))
    out.append(("integers", r.integers(-2, 3, (n, n)).astype(float), r.integers(-2, 3, n).astype(float)))
    out.append(("high words", r.choice([-1.0, 1.0], (n, n)) * (1 + r.integers(0, 4, (n, n)) * 2.0 ** -50), g(n)))
    z = g(n, n)
    z[:, r.integers(n)] = 0.0
    out.append(("zero column", z, g(n)))
    out.append(("zeros", np.zeros((n, n)), g(n)))
    out.append(("negative zeros", np.where(r.random((n, n)) < 0.5, -0.0, g(n, n)) + 3 * np.eye(n),
                np.where(r.random(n) < 0.5, -0.0, g(n))))
    out.append(("zero right-hand side", g(n, n), np.zeros(n)))
    for name, v in (("nan", np.nan), ("inf", np.inf)):
        for where in ("diagonal", "below", "above"):
            a = g(n, n)
            i, j = sorted(r.integers(n, size=2))
            a[(i, i) if where == "diagonal" else (j, i) if where == "below" else (i, j)] = v
            out.append((f"{name} {where}", a, g(n)))
        b = g(n)
        b[r.integers(n)] = v
        out.append((f"{name} on the right", g(n, n), b))
    for e in (401, 399, 600, 900, -399, -401, -600, -900, -1040):
        out.append((f"scale {e}", g(n, n) * 2.0 ** e, g(n)))
        out.append((f"right-hand side {e}", g(n, n), g(n) * 2.0 ** e))
    out.append(("rows apart", np.ldexp(g(n, n), r.integers(-450, 450, (n, 1))), g(n)))
    out.append(("columns apart", np.ldexp(g(n, n), r.integers(-450, 450, (1, n))), g(n)))
    out.append(("entries apart", np.ldexp(g(n, n), r.integers(-60, 60, (n, n))), g(n)))
    return out


def reference(A, b):
    """LU with its rows at their positions, the row gather, x."""
    n = len(b)
    F, x = np.ascontiguousarray(A).copy(), np.ascontiguousarray(b).copy()
    piv = (ctypes.c_int * n)()
    d = ctypes.POINTER(ctypes.c_double)
    O.lib().oo_lu_solve(n, F.ctypes.data_as(d), piv, x.ctypes.data_as(d))
    perm = np.arange(n)
    for k in range(n):
        perm[[k, piv[k]]] = perm[[piv[k], k]]
    return F, perm, x


def same(a, b):
    """Bits, but for the sign and payload of a NaN."""
    return ((a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b))).all()


def test_lds_fits():
    for nmax, ns in SIZES.items():
        for n in ns:
            assert n <= nmax and lds_bytes(n, n | 1) <= MAX_LDS and lds_bytes(n, nmax | 1) <= MAX_LDS
            # reads past the last row's end (up to 7 entries) stay inside
            assert (n * (n | 1) + 7) * 8 <= lds_bytes(n, n | 1)


@pytest.mark.gpu
@pytest.mark.parametrize("threads", [256, 512])
@pytest.mark.parametrize("nmax", sorted(SIZES))
def test_lu_bits(nmax, threads):
    _lib.load()
    import torch
    torch.cuda.synchronize()
    with open("/proc/self/maps") as f:   # the HIP runtime that torch brought
        hip = ctypes.CDLL(next(l.split()[-1] for l in f if "libamdhip64" in l))
    co = os.path.join(os.path.dirname(_lib.LIB_PATH), f"devcheck_lu_{nmax}.co")
    mod, fn = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipModuleLoad(ctypes.byref(mod), co.encode()) == 0, co
    assert hip.hipModuleGetFunction(ctypes.byref(fn), mod, b"lu_check") == 0
    for n in SIZES[nmax]:
        cases = matrices(n)
        m = len(cases)
        A = torch.as_tensor(np.stack([c[1] for c in cases])).cuda()
        b = torch.as_tensor(np.stack([c[2] for c in cases])).cuda()
        refs = [reference(c[1], c[2]) for c in cases]
        for ld in sorted({n | 1, nmax | 1}):
            print(f"[case] lu n {n} ld {ld} threads {threads}", flush=True)
            LU, x, xneg = torch.empty_like(A), torch.empty_like(b), torch.empty_like(b)
            perm = torch.empty(m, n, dtype=torch.int32, device=A.device)
            vals = [ctypes.c_void_p(A.data_ptr()), ctypes.c_void_p(b.data_ptr()), ctypes.c_int(n), ctypes.c_int(ld),
                    *(ctypes.c_void_p(t.data_ptr()) for t in (LU, perm, x, xneg))]
            args = (ctypes.c_void_p * len(vals))(*(ctypes.addressof(v) for v in vals))
            torch.cuda.synchronize()
            assert hip.hipModuleLaunchKernel(fn, m, 1, 1, threads, 1, 1, lds_bytes(n, ld), None, args, None) == 0
            torch.cuda.synchronize()
            LUh, ph, xh, gh = (t.cpu().numpy() for t in (LU, perm, x, xneg))
            for (name, _, _), (F, pr, xr), f, p, xx, gg in zip(cases, refs, LUh, ph, xh, gh):
                assert np.array_equal(p, pr), (n, ld, name)
                assert same(f, F), (n, ld, name)
                assert same(xx, xr) and same(gg, -xr), (n, ld, name)
    assert hip.hipModuleUnload(mod) == 0
