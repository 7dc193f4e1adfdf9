"""The library on a HIP runtime without a GPU (fake_hip.cpp), for tests of its
host code in a process of their own: which kernel a call launches, what it
allocates and what it does without memory or under capture.  No kernel runs."""
import ctypes
import os
import subprocess
import sys
import types

import numpy as np  # noqa: F401  (for the bodies)

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))


def run(body, tmp_path):
    """Runs `body` (statements; aa, fake, Tensor and Stream at hand) in a new process."""
    so = tmp_path / "fake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wl,-soname,libamdhip64.so.7", "-o", str(so),
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    script = tmp_path / "body.py"
    script.write_text("from host_library import *\naa, fake = load(%r)\n%s" % (str(so), body))
    env = dict(os.environ, PYTHONPATH=HERE)
    done = subprocess.run([sys.executable, str(script)], env=env, capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout + done.stderr
    return done.stdout


class Stream:
    def __init__(self, handle=0):
        self.cuda_stream = handle


class Tensor:
    """Memory with the few tensor methods that the library's Python side reads."""
    is_cuda, device = True, "cuda:0"

    def __init__(self, shape, size=4, dtype="float32"):
        self.shape, self.size, self.dtype = tuple(shape), size, dtype
        n = size
        for s in shape:
            n *= s
        self.buffer = ctypes.create_string_buffer(n + 256)
        self.at = (ctypes.addressof(self.buffer) + 255) // 256 * 256

    def is_contiguous(self):
        return True

    def dim(self):
        return len(self.shape)

    def data_ptr(self):
        return self.at

    def element_size(self):
        return self.size

    def stride(self, dim):
        return self.shape[1] if dim == 0 else 1


class Fake:
    def __init__(self, lib):
        self.lib = lib
        lib.fake_device_bytes.restype = lib.fake_blocks.restype = lib.fake_block.restype = ctypes.c_size_t
        lib.fake_block.argtypes = [ctypes.c_size_t]
        lib.fake_launch_name.restype = ctypes.c_char_p
        lib.fake_launch_stream.restype = ctypes.c_void_p
        lib.fake_launch_word.restype = ctypes.c_uint64
        lib.fake_fail_allocations.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
        lib.fake_fail_host_allocations.argtypes = [ctypes.c_size_t]
        lib.fake_allocated.restype = ctypes.c_size_t
        lib.fake_capture.argtypes = [ctypes.c_void_p]
        lib.fake_cost.argtypes = [ctypes.c_char_p, ctypes.c_float]

    def kernels(self):
        """Names of the kernels launched since the last call."""
        names = [self.lib.fake_launch_name(i).decode() for i in range(self.lib.fake_launches())]
        self.lib.fake_clear_launches()
        return names

    def argument_words(self, part, word):
        """The given 8-byte word of the first argument of every launch of `part` since kernels()."""
        return [self.lib.fake_launch_word(i, word) for i in range(self.lib.fake_launches())
                if part in self.lib.fake_launch_name(i).decode()]

    def ran(self, part):
        return any(part in n for n in self.kernels())

    def blocks(self):
        """Numbers of the device blocks in use."""
        return [self.lib.fake_block(i) for i in range(self.lib.fake_blocks())]

    def allocations(self):
        return [self.lib.fake_allocated(i) for i in range(self.lib.fake_allocations())]

    def fail_allocations(self, low=2 ** 64 - 1, high=2 ** 64 - 1):
        """Device allocations of low <= bytes < high fail; without arguments none do."""
        self.lib.fake_fail_allocations(low, high)


def load(so):
    fake = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    torch = types.ModuleType("torch")   # the real one would load the real runtime
    for name, size in (("uint8", 1), ("float32", 4), ("float64", 8)):
        setattr(torch, name, name)
    torch.empty = lambda shape, dtype, device: Tensor(shape if isinstance(shape, tuple) else (shape,),
                                                      {"uint8": 1, "float32": 4, "float64": 8}[dtype], dtype)
    torch.cuda = types.SimpleNamespace(current_stream=lambda *a: Stream())
    sys.modules["torch"] = torch
    for p in ("astro-accelerate_amd", "oracle"):
        sys.path.insert(0, os.path.join(ROOT, p))
    import py_astro_accelerate as aa
    aa.load_library()
    return aa, Fake(fake)
