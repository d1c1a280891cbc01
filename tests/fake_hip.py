"""The host code of librender_hip on the CPU: its HIP calls end in a stand-in runtime (fake_hip.cpp) that
writes them down and can make a chosen one fail.  No kernel runs, so results are never looked at;
the order of calls and the error paths are.

A test runs its body in a process of its own (``child``), since the library keeps one state and the
stand-in must be loaded before it.
"""
import ctypes
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def build(folder) -> str:
    """Compiles the stand-in into `folder`; its path."""
    out = os.path.join(str(folder), "libfakehip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-I/opt/rocm/include", "-o", out,
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    return out


def child(fake: str, module: str, function: str, *args) -> None:
    """module.function(hip, *args) in a process whose HIP runtime is `fake`; its failures are raised here."""
    code = (f"import sys; sys.path[:0] = [{HERE!r}, {ROOT!r}]\n"
            f"import fake_hip\nhip = fake_hip.Fake({fake!r})\n"
            f"import {module}\n{module}.{function}(hip, *{args!r})\nprint('CHILD DONE', flush=True)\n"
            f"import os; os._exit(0)\n")
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and p.stdout.endswith("CHILD DONE\n"), (p.returncode, p.stdout[-2000:], p.stderr[-4000:])


class Fake:
    """The stand-in in this process, to be loaded before librender_hip."""

    def __init__(self, path: str):
        self.lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        self.lib.fake_lines.restype = ctypes.c_char_p
        self.lib.fake_fail.argtypes = [ctypes.c_char_p, ctypes.c_int]

    def lines(self) -> list:
        """The calls since the last clear()."""
        return self.lib.fake_lines().decode().splitlines()

    def clear(self) -> None:
        self.lib.fake_clear()

    def fail(self, what: str, nth: int = 1) -> None:
        """The nth call from here whose line contains `what` fails."""
        self.lib.fake_fail(what.encode(), nth)

    def device(self, nbytes: int) -> int:
        p = ctypes.c_void_p()
        assert self.lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes)) == 0
        return p.value

    def page_locked(self, nbytes: int) -> int:
        p = ctypes.c_void_p()
        assert self.lib.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes), 0) == 0
        return p.value
