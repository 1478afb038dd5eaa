"""The calls from Python (``research_amd/csrc/host_calls.cpp``) on the CPU: the checks against what they stand for, the arguments that the
library's functions take, and what is refused."""

import re
import subprocess
import sys
import sysconfig

import pytest
import torch

from research_amd import _host as host
from research_amd import _lib, ops

_lib.load()


def test_a_module_that_is_built_after_the_import():
    """``ops`` imported while there is no native module: calls say so, and work once there is one."""
    code = """
import sys
import sysconfig
class Missing:
    def find_spec(self, name, path=None, target=None):
        if name == "research_amd._host":
            raise ImportError("not built")
sys.meta_path.insert(0, Missing())
import torch
from research_amd import ops
a = torch.zeros(3, 8)
for call in (lambda: ops._typed(torch.float32, a), lambda: ops.softcap(a, 1.0)):
    try:
        call()
    except FileNotFoundError as e:
        assert "research_amd.build" in str(e)
    else:
        raise SystemExit("not refused")
del sys.meta_path[0]
assert ops._shaped(a, 3, 8) is True and ops._row_stride(a) == 8
for bad, error in ((lambda: ops._typed(torch.int32, a), ValueError), (lambda: ops._dense(a.t()), ValueError), (lambda: ops.softcap(a, 1.0), RuntimeError)):
    try:
        bad()
    except error:
        pass
    else:
        raise SystemExit("not refused")
ops._run("pa_softcap", a, None, 0, 1.0, 0, None)
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=ops.__file__.rsplit("/research_amd/", 1)[0])


def test_checks():
    a, b = torch.zeros(3, 8), torch.zeros(4, 6, dtype=torch.int32)
    host.dense(a, None, b, a[1:], torch.nn.Parameter(a))
    with pytest.raises(ValueError, match="contiguous"):
        host.dense(None, b, a[:, 1:])
    host.typed(torch.float32, a, None, a[:, 1:])
    with pytest.raises(ValueError, match="expected torch.float32, got torch.int32"):
        host.typed(torch.float32, None, a, b)
    assert host.nbytes(None) == 0 and host.nbytes(b) == 96 and host.nbytes(a[:, 1:3].to(torch.bfloat16)) == 12
    assert host.shaped(a, 3, 8) and host.shaped(a, None, 8) and not host.shaped(a, 3, 7) and not host.shaped(a, 3) and not host.shaped(a, 3, 8, 1)
    assert host.shaped(torch.zeros(()),) and host.shaped(torch.zeros(0, 2), 0, None)
    for bad in (3, "x", None):
        with pytest.raises(TypeError):
            host.shaped(bad, 1)
        with pytest.raises(TypeError):
            host.dense(a, bad if bad is not None else 1.0)
    with pytest.raises(RuntimeError, match="HIP device"):
        host.stream(a)


@pytest.mark.parametrize("t", [torch.zeros(3, 8), torch.zeros(3, 8)[:, 2:5], torch.zeros(1, 8), torch.zeros(1, 8)[:, :3], torch.zeros(5, 1),
                               torch.zeros(8, 5)[:, :1], torch.zeros(0, 4), torch.zeros(4, 0), torch.zeros(4, 3).t(), torch.zeros(1, 4, 3)[0].t()[:, :1],
                               torch.zeros(3, 8)[::2], torch.zeros(8)[None].expand(3, 8), torch.zeros(3), torch.zeros(2, 3, 4), torch.zeros(3, 8)[:, ::2]])
def test_row_stride(t):
    want = None
    if t.dim() == 2:
        (rows, cols), (row, col) = t.shape, t.stride()
        if cols <= 1 or col == 1:
            want = row if rows > 1 else max(row, cols)
    if want is None:
        with pytest.raises(ValueError, match="contiguous rows"):
            host.row_stride(t)
    else:
        assert host.row_stride(t) == want


def test_every_call_takes_what_the_library_declares():
    source = open(ops.__file__).read()
    names = set(re.findall(r'_run\("(pa_\w+)"', source)) | {"pa_decode", "pa_decode_split", "pa_decode_reduce", "pa_prefill_paged"}
    assert len(names) > 30
    for name in names:
        with pytest.raises(TypeError, match=f"takes {len(_lib.SIGNATURES[name][1])} arguments, got 0"):
            getattr(host, name)()


def test_arguments():
    lib = _lib.load()
    assert host.pa_moe_workspace_bytes(1000, 64, 8) == lib.pa_moe_workspace_bytes(1000, 64, 8) > 0
    assert host.pa_moe_workspace_bytes(1000, 64 + (1 << 32), True) == lib.pa_moe_workspace_bytes(1000, 64, 1)  # (integers wrap, as in ctypes)
    for bad in (1.5, None, "8", torch.zeros(1)):
        with pytest.raises(TypeError):
            host.pa_moe_workspace_bytes(1000, 64, bad)
    t = torch.zeros(4)
    call = lambda x, out, n, cap: host.pa_softcap(x, out, n, cap, 0, None)
    assert call(t, None, 0, 1.0) == 0 and call(t.data_ptr(), t, 0, 1) == 0  # (nothing to do)
    assert call(t, t, -1, 1.0) == _lib.PA_ERR_INVALID_ARG and "softcap" in _lib.last_error()
    for bad in (1.5, "x", [t]):
        with pytest.raises(TypeError):
            call(bad, t, 0, 1.0)
    with pytest.raises(TypeError):
        call(t, t, 0, "1")


@pytest.mark.parametrize("name,count", [("gated_linear", 25), ("delta_rule", 20), ("channel_linear", 17), ("lightning", 13), ("narrow_linear", 2), ("moe_choose", 12),
                                        ("moe_product", 9)])
def test_whole_calls_that_do_not_fit_are_left_to_the_wrapper(name, count):
    """Another number of arguments, arguments of other kinds and tensors that lie on no device: no answer, and no exception."""
    call = getattr(host, name)
    t = torch.zeros(4, 4)
    for args in ((), (t,) * (count - 1), (t,) * count, (1,) * count, (1.0,) * count, (None,) * count, ("x",) * count, (1 << 70,) * count, (-1,) * count):
        assert call(*args) is None
    for i in range(count):
        assert call(*(t if j == i else 1 for j in range(count))) is None and call(*(1.0 if j == i else t for j in range(count))) is None


def test_whole_calls_on_the_cpu_say_what_the_wrapper_says():
    i32 = lambda *n: torch.zeros(*n, dtype=torch.int32)
    runs = ops.Portions(i32(2), i32(2))
    rows = torch.zeros(2, 64)
    for call in (lambda: ops.narrow_linear(rows, torch.zeros(3, 64)), lambda: ops.moe_choose(rows, 64, 2, 1, 1),
                 lambda: ops.lightning(torch.zeros(2, 192), runs, torch.zeros(2, 1, 64, 64), torch.zeros(1, 65), 1, 64, 64, rows),
                 lambda: ops.channel_linear(rows, rows, rows, None, torch.zeros(64), runs, torch.zeros(2, 1, 64, 64), 1, 64, 64, rows.clone())):
        with pytest.raises(RuntimeError, match="HIP device"):
            call()
    for call in (lambda: ops.narrow_linear(rows, torch.zeros(3, 63)), lambda: ops.narrow_linear(rows, torch.zeros(64, 3).t()), lambda: ops.moe_choose(rows, 63, 2, 1, 1),
                 lambda: ops.moe_choose(rows.bfloat16(), 64, 2, 1, 1),
                 lambda: ops.lightning(torch.zeros(2, 192), runs, torch.zeros(2, 1, 64, 48), torch.zeros(1, 65), 1, 64, 64, rows),
                 lambda: ops.channel_linear(rows, rows[:, :32], rows, None, torch.zeros(64), runs, torch.zeros(2, 1, 64, 64), 1, 64, 64, rows.clone())):
        with pytest.raises(ValueError):
            call()


def test_a_module_of_another_interpreter_or_torch_is_not_taken():
    root = ops.__file__.rsplit("/research_amd/", 1)[0]
    assert host.__file__.endswith("_host" + sysconfig.get_config_var("EXT_SUFFIX"))  # (which other interpreters do not look for)
    code = """
import torch.version
torch.version.__version__ = "1.0"
try:
    import research_amd._host
except ImportError as e:
    assert "torch 1.0" in str(e), e
else:
    raise SystemExit("taken")
from research_amd import _lib
try:
    _lib.load()
except FileNotFoundError as e:
    assert "research_amd.build" in str(e)
else:
    raise SystemExit("taken")
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=root)
    rules = lambda *args: subprocess.run(["make", "-C", root + "/research_amd/csrc", "-n", f"PYTHON={sys.executable}", *args, "host"], check=True,
                                         stdout=subprocess.PIPE, text=True).stdout
    assert "host_calls.cpp" in rules("TORCH_VERSION=1.0")  # (another torch than it was built for: built again)
