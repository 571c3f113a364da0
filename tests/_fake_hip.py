"""The library's host code on a machine without a GPU: runs a script in a process of its own whose HIP calls end in
tests/cxx/fake_hip.c.  Its tensors claim to be on the GPU and hold host memory; kernels are counted and not run."""
import ctypes
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(tmp_path, script, first=""):
    """Runs `first`, then the script after `from _fake_hip import *` (and _lib); fails with its output if it does not end well."""
    lib = os.path.join(str(tmp_path), "libfake_hip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-fexceptions", "-o", lib, os.path.join(ROOT, "tests", "cxx", "fake_hip.c"),
                    "-l:libstdc++.so.6"], check=True)
    path = os.pathsep.join([ROOT, os.path.join(ROOT, "tests"), os.environ.get("PYTHONPATH", "")])
    p = subprocess.run([sys.executable, "-c", first + "\nfrom _fake_hip import *\nfrom _fake_hip import _lib\n" + script], text=True, timeout=300, cwd=str(tmp_path),
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, env=dict(os.environ, PYTHONPATH=path, FAKE_HIP=lib))
    assert p.returncode == 0, "exit %d\n%s" % (p.returncode, p.stdout[-6000:])
    return p.stdout


if os.environ.get("FAKE_HIP"):                           # in the script's process, ahead of torch
    hip = ctypes.CDLL(os.environ["FAKE_HIP"], mode=ctypes.RTLD_GLOBAL)

    import torch

    torch.cuda._lazy_init = lambda: None
    torch.cuda.synchronize = lambda *a: None
    from cuv_amd import _lib, dia as D

    L = _lib.lib()

    def flag(name, value=None, kind=ctypes.c_int):
        """Reads or sets a variable of fake_hip.c."""
        v = kind.in_dll(hip, name)
        if value is not None:
            v.value = value
        return v.value

    class _DLTensor(ctypes.Structure):                   # DLPack's DLManagedTensor, its tensor's fields in place
        _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int), ("device_id", ctypes.c_int), ("ndim", ctypes.c_int),
                    ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16),
                    ("shape", ctypes.POINTER(ctypes.c_int64)), ("strides", ctypes.POINTER(ctypes.c_int64)),
                    ("byte_offset", ctypes.c_uint64), ("ctx", ctypes.c_void_p), ("deleter", ctypes.c_void_p)]

    _capsule = ctypes.pythonapi.PyCapsule_New
    _capsule.restype, _capsule.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
    _keep = []

    def tensor(*shape, bytes_at=None):
        """A float32 tensor on cuda:0 that lies in host memory; bytes_at: at that address instead, never touched."""
        n = 1
        for s in shape:
            n *= s
        buf = (ctypes.c_float * (n if bytes_at is None else 1))()
        dims = (ctypes.c_int64 * len(shape))(*shape)
        m = _DLTensor(bytes_at or ctypes.addressof(buf), 10, 0, len(shape), 2, 32, 1, dims, None, 0, None, None)
        _keep.append((buf, dims, m))
        return torch.utils.dlpack.from_dlpack(_capsule(ctypes.addressof(m), b"dltensor", None))

    class _Matrix(D.dev_dia_matrix_f):
        def alloc(self):
            self.vec = tensor(self.num_dia * self.stride, bytes_at=1 << 40)

        @property
        def desc(self):
            if self._desc is None:
                d = ctypes.c_void_p()
                _lib.check(L.cuvdia_desc_create(ctypes.byref(d), self._offsets.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                                                self.num_dia, self.h, self.w, self.stride, self.row_fact), "cuvdia_desc_create")
                self._desc, self._desc_ptr = d, d.value
            return self._desc

    def matrix(h, w, offsets, row_fact=1):
        m = _Matrix(h, w, len(offsets), max(h, w), row_fact)
        m.set_offsets(offsets)
        m.desc
        return m
