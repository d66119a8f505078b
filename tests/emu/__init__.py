"""The island resolver's device code built for the CPU (islands.cpp), one
workgroup as fibers, for what a device run cannot be asked: accesses out of
bounds, other orders of the waves, and worlds that find no room in the log."""
import ctypes
import os
import re
import subprocess

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
CSRC = os.path.join(ROOT, "cubez_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"

PLAIN, LABEL, MAT = 0, 1, 3
POS_VEL = 3
BODY = {"pos": 3, "quat": 4, "vel": 3, "rot": 3, "inv_mass": 1, "iit_body": 9, "iit_world": 9, "transform": 12,
        "last_acc": 3, "motion": 1, "flags": 0}
CONTACT = {"body0": 0, "body1": 0, "point": 3, "normal": 3, "pen": 1, "c2w": 9, "rel": 6, "cvel": 3, "ddv": 1,
           "fric": 1, "rest": 1}


class _World(ctypes.Structure):
    _fields_ = ([(k, ctypes.c_int32) for k in ("n", "C", "kind", "mode", "f64", "across", "threads")]
                + [(k, ctypes.c_int64) for k in ("mult", "fixed", "log_cap", "max_steps")]
                + [("dt", ctypes.c_double)]
                + [(k, ctypes.c_void_p) for k in (*BODY, *CONTACT, "labels", "iters", "left")])


def build(out_dir, optimise="-O1"):
    """The headers without their launches and inline assembly, and the library
    (with -O0, every access of the source is made)."""
    for name in os.listdir(CSRC):
        if not name.endswith(".h"):
            continue
        with open(os.path.join(CSRC, name)) as f:
            s = f.read()
        s = re.sub(r"[\w<>, ():]+<<<[^;]*;", ";", s)
        s = re.sub(r'asm volatile\("" : "\+v"\([^;]*;', ";", s)
        s = s.replace("extern __shared__ __align__(16) char isl_lds[];", "")
        with open(os.path.join(out_dir, name), "w") as f:
            f.write(s)
    lib = os.path.join(out_dir, "libislands.so")
    subprocess.run([CLANG, optimise, "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-w", "-I", HERE,
                    "-I", out_dir, "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "islands.cpp"), "-o", lib],
                   check=True)
    return ctypes.CDLL(lib)


def _planes(x, k, real):
    return np.array(np.asarray(x).reshape(-1, k).T, real, order="C")


def resolve(lib, o, contacts, dt, mult=4, fixed=0, precision="f64", kind=PLAIN, log_cap=200000, across=False, threads=256):
    """ResolveContacts of an oracle world's state and contact list.  Returns the
    status (0), the arrays after it ([plane][n]), the iterations of both phases
    and how many worlds were handed to the serial kernel."""
    real = np.float64 if precision == "f64" else np.float32
    n, C = o.n, len(contacts)
    src = {"fric": "friction", "rest": "restitution"}
    out = {k: _planes(o.a[k], w, real) if w else o.a[k].copy() for k, w in BODY.items()}
    for k, w in CONTACT.items():
        if w == 0:
            out[k] = contacts[k].astype(np.int32)
        elif k in ("c2w", "rel", "cvel", "ddv"):
            out[k] = np.zeros((w, C), real)
        else:
            out[k] = _planes(contacts[src.get(k, k)], w, real)
    out["labels"] = np.zeros((C, 13), np.float32)
    iters, left = np.zeros(2, np.int64), np.zeros(1, np.int32)
    q = _World(n, C, kind, POS_VEL | (4 if kind == LABEL else 0), precision == "f64", across, threads, mult, fixed, log_cap,
               50_000_000, dt)
    for k in (*BODY, *CONTACT, "labels"):
        setattr(q, k, out[k].ctypes.data)
    q.iters, q.left = iters.ctypes.data, left.ctypes.data
    rc = lib.emu_resolve(ctypes.byref(q))
    return rc, out, tuple(int(i) for i in iters), int(left[0])
