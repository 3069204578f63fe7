"""A context that interpreter exit finalizes before its systems stays usable by their finalizers."""
import subprocess
import sys

CODE = """
import ctypes, sys
sys.path.insert(0, {root!r})
from vfvm import _capi
order = []
class Lib:
    def vfvm_ctx_destroy(self, h):
        order.append("ctx"); print("ctx", flush=True)
_capi._LIB = Lib()
class System:
    def __init__(self, ctx):
        self.ctx = ctx; self.me = self
    def __del__(self):
        print("system" if "ctx" not in order else "system after its context", flush=True)
ctx = _capi.Context.__new__(_capi.Context)
ctx.handle = 1
if {cycle}:
    ctx.me = ctx
keep = System(ctx)
def f(): return keep
if not {cycle}:
    keep.me = None
    del keep, ctx
"""


def _run(cycle):
    import conftest
    code = CODE.format(root=conftest.ROOT + "/voronoifvm.jl_amd", cycle=cycle)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return r.stdout.split("\n")


def test_exit_keeps_the_context():
    assert "system after its context" not in _run(True)


def test_a_dropped_context_is_destroyed():
    assert _run(False)[:2] == ["system", "ctx"]
