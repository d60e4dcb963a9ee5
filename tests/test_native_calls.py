"""The native calls (csrc/binding.cpp) decline what is no plain call, before
any effect, so that the Python code behind them answers as it always did."""

from __future__ import annotations

import glob
import os
import shutil
import subprocess
import sys
import threading
import time

import pytest
import torch

from conftest import ROOT
from elysium_wan_amd import _lib

PACKAGE = os.path.join(ROOT, "elysium_wan_amd")
LIBRARIES = ("libelyhip.so", "_native.so")


class _Sub(torch.Tensor):
    pass


def _declined(x):
    N = _lib.load_native()
    return [N.quantize(x, "e4m3", False), N.roundtrip(x, "e4m3", True), N.cast_bf16(x), N.widen_bf16(x), N.fold_add(x, x),
            N.dequantize(x, x, True), N.clip([x], 1.0)]


def test_host_tensors_and_other_objects_are_declined():
    for x in (torch.zeros(3, 8), torch.zeros(3, 8, dtype=torch.float16), None, 3.0, "x"):
        assert all(r is None for r in _declined(x))
    p = torch.zeros(4)
    args = [[p], [torch.ones(4)], None, {}, torch.zeros(1), None, 0, 0, 0, None, None, lambda t: [0.0] * 8]
    assert _lib.load_native().adamw_step(*args) is None and float(args[4][0]) == 0.0


def _copy_of_the_package(tmp_path, *names):
    d = tmp_path / "elysium_wan_amd"
    d.mkdir()
    for f in glob.glob(os.path.join(PACKAGE, "*.py")) + [os.path.join(PACKAGE, n) for n in names]:
        shutil.copy(f, d)
    return d


def _run(tmp_path, code):
    r = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True, text=True, timeout=120,
                       env={**os.environ, "PYTHONDONTWRITEBYTECODE": "1"})
    assert r.returncode == 0, r.stdout + r.stderr


def test_a_library_built_after_the_import_is_used(tmp_path):
    """Nothing built: host calls answer as they do with the libraries, the
    rest say what is missing; once the libraries are there, they load."""
    _copy_of_the_package(tmp_path)
    _run(tmp_path, f"""
import shutil, torch
from elysium_wan_amd import _lib, fp8, optim, pieces

n = torch.tensor([3])
pieces.fold_add(n, torch.tensor([4]))
assert int(n) == 7 and float(optim.clip_grad_norm_([torch.zeros(2)], 1.0)) == 0.0
for call, error in ((lambda: fp8.quantize(torch.zeros(2, 8)), ValueError), (lambda: pieces.cast_piece(torch.zeros(8), torch.bfloat16), ValueError),
                    (lambda: _lib.workspace(torch.device("cuda", 0), 1), RuntimeError), (lambda: _lib.load(), RuntimeError)):
    try:
        call()
    except error as e:
        assert "GPU" in str(e) or "build the HIP library" in str(e), e
    else:
        raise AssertionError("not refused")
shutil.copy({os.path.join(PACKAGE, LIBRARIES[0])!r}, "elysium_wan_amd")
try:
    _lib.load_native()
except RuntimeError as e:
    assert "build the HIP library" in str(e), e
else:
    raise AssertionError("loaded without its file")
shutil.copy({os.path.join(PACKAGE, LIBRARIES[1])!r}, "elysium_wan_amd")
assert _lib.load_native().quantize(torch.zeros(2, 8), "e4m3", False) is None and _lib.load().ely_abi_version() == 1
""")


# as a rebuild leaves the files: new ones at the old paths
REPLACE = """
import os, shutil
def replaced(name, new):
    shutil.copy(new, "new")
    os.replace("new", "elysium_wan_amd/" + name)
def mapped(name):
    return {line.split()[4] for line in open("/proc/self/maps") if "/elysium_wan_amd/" in line and line.rstrip().endswith(name)}
"""


@pytest.mark.parametrize("first", ["load", "load_native"])
def test_a_library_rebuilt_after_the_import_is_the_one_that_runs(tmp_path, first):
    """The new library answers through ctypes and through the new _native, and
    a later rebuild changes nothing for this process."""
    _copy_of_the_package(tmp_path, *LIBRARIES)
    stub = tmp_path / "stub.c"
    stub.write_text("\n".join(f"int {n}(void) {{ return {77 if n == 'ely_abi_version' else 0}; }}" for n in _lib.EXPORTS))
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "stub.so"), str(stub)], check=True)
    _run(tmp_path, REPLACE + f"""
import elysium_wan_amd
from elysium_wan_amd import _lib, accumulate, boundary, f32_planes, fp8, fp8_planes, optim, pieces, planes
replaced("libelyhip.so", "stub.so")
replaced("_native.so", {os.path.join(PACKAGE, "_native.so")!r})
_lib.{first}()
N = _lib.load_native()
assert _lib.load().ely_abi_version() == 77 and N.abi_version() == 77
for name in ("libelyhip.so", "_native.so"):
    assert str(os.stat("elysium_wan_amd/" + name).st_ino) in mapped(name), name
replaced("libelyhip.so", {os.path.join(PACKAGE, "libelyhip.so")!r})
assert _lib.load().ely_abi_version() == 77 and _lib.load_native() is N
""")


def test_an_unchanged_library_is_mapped_once(tmp_path):
    _copy_of_the_package(tmp_path, *LIBRARIES)
    _run(tmp_path, REPLACE + """
from elysium_wan_amd import _lib
N = _lib.load_native()
assert N.abi_version() == _lib.load().ely_abi_version() == 1
for name in ("libelyhip.so", "_native.so"):
    assert mapped(name) == {str(os.stat("elysium_wan_amd/" + name).st_ino)}, name
""")


@pytest.mark.gpu
def test_plain_calls_are_taken_and_equal_the_python_path(monkeypatch):
    from elysium_wan_amd import fp8, optim, pieces

    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(33, 1001, generator=g, device="cuda").bfloat16()
    long = torch.randn(1, 70001, generator=g, device="cuda")

    def calls():
        q, k = fp8.quantize(x)
        ql, kl = fp8.quantize(long, "e5m2", per_tensor=True)
        acc = x.float()
        pieces.fold_add(acc, x)
        h = x.clone()
        pieces.fold_add(h, x)
        ps = [x.float().requires_grad_(True), long.clone().requires_grad_(True)]
        opt = optim.FusedAdamW(ps, lr=1e-3, weight_decay=0.1, max_norm=1.0, working_copy=True)
        for gs in ([x, long], [None, long.bfloat16()], [x.float(), long.bfloat16()]):  # state made, one skipped, two dtypes
            opt.step(grads=gs)
            opt.step(grads=tuple(gs), acc=[torch.ones_like(p) for p in ps])
        cs = [torch.zeros_like(long), torch.zeros_like(x), torch.zeros(3, device="cuda")]
        cs[0].grad, cs[1].grad = long.clone(), x.clone()
        total = optim.clip_grad_norm_(iter(cs), 0.5)
        return [q.view(torch.uint8), k, ql.view(torch.uint8), kl, fp8.roundtrip(x, "e5m2"), fp8.roundtrip(long, per_tensor=True),
                fp8.dequantize(q, k), fp8.dequantize(ql, kl, torch.bfloat16), pieces.cast_piece(long, torch.bfloat16),
                pieces.fold_start(x), acc, h, *[p.detach() for p in ps], *opt.working_copies, opt.grad_norm(),
                *[opt.state[i][n] for i in (0, 1) for n in ("step", "exp_avg", "exp_avg_sq")], total, cs[0].grad, cs[1].grad]

    N = _lib.load_native()
    taken = []

    class Spy:
        def __getattr__(self, name):
            f = getattr(N, name)

            def call(*a):
                r = f(*a)
                taken.append((name, r is not None))
                return r

            return f if name == "workspace" else call

    class Off:
        workspace = staticmethod(N.workspace)

        def __getattr__(self, name):
            return lambda *a: None

    monkeypatch.setattr(_lib, "_native", Spy())
    fast = calls()
    # the optimizer's first step, which makes its state, does not ask; every call that does is taken
    assert all(ok for _, ok in taken) and [n for n, _ in taken].count("adamw_step") == 5
    assert {n for n, ok in taken if ok} == {"quantize", "roundtrip", "dequantize", "cast_bf16", "widen_bf16", "fold_add", "adamw_step", "clip"}
    monkeypatch.setattr(_lib, "_native", Off())
    slow = calls()
    for a, b in zip(fast, slow):
        assert a.dtype == b.dtype and a.shape == b.shape and a.device == b.device and torch.equal(a, b)


@pytest.mark.gpu
def test_views_wrappers_and_modes_are_declined():
    from torch.overrides import TorchFunctionMode

    x = torch.randn(16, 32, device="cuda").bfloat16()
    N = _lib.load_native()
    for y in (x.t(), x.to(torch.float16), x[0, 0], x[:0], x.as_subclass(_Sub), x.cpu()):
        assert N.quantize(y, "e4m3", False) is None and N.roundtrip(y, "e4m3", False) is None
    assert N.quantize(x, "e3m4", False) is None and N.quantize(x, 3, False) is None
    assert N.fold_add(x.float().t(), x) is None and N.fold_add(x.float(), x[:3]) is None
    q, k = N.quantize(x, "e4m3", False)
    assert N.dequantize(q, k[:3], True) is None and N.dequantize(q, k.long(), True) is None and N.dequantize(x, k, True) is None
    seen = []
    torch.vmap(lambda row: seen.append(N.roundtrip(row, "e4m3", False)) or row * 1)(x)
    with TorchFunctionMode():
        seen.append(N.quantize(x, "e4m3", False))
    with torch._subclasses.FakeTensorMode(allow_non_fake_inputs=True):
        seen.append(N.quantize(x, "e4m3", False))
    assert seen == [None, None, None]


@pytest.mark.gpu
def test_a_failed_check_leaves_state_and_tensors_alone():
    """The native step looks every tensor over before it counts a step."""
    from elysium_wan_amd import optim

    ps = [torch.ones(300, device="cuda", requires_grad=True) for _ in range(3)]
    opt = optim.FusedAdamW(ps, lr=1e-3, max_norm=1.0)
    good = [torch.ones(300, device="cuda") for _ in ps]
    opt.step(grads=good)
    before = [p.detach().clone() for p in ps]
    for bad in (torch.ones(299, device="cuda"), torch.ones(600, device="cuda")[::2], torch.ones(300), torch.ones(300, device="cuda").half()):
        with pytest.raises(ValueError):
            opt.step(grads=good[:2] + [bad])
        assert [float(opt.state[i]["step"]) for i in range(3)] == [1.0] * 3
        assert all(torch.equal(p.detach(), b) for p, b in zip(ps, before))


@pytest.mark.gpu
def test_the_clips_total_is_a_tensor_of_its_own():
    """As the Python path's clone: no view, which could not be detached in place."""
    from elysium_wan_amd import optim

    p = torch.zeros(300, device="cuda")
    p.grad = torch.full((300,), 2.0, device="cuda")
    total = optim.clip_grad_norm_([p], 1.0)
    assert not total._is_view() and total.dim() == 0 and total.dtype == torch.float32
    total.detach_()
    again = optim.clip_grad_norm_([p], 1.0)
    assert abs(float(total) - 2.0 * 300**0.5) < 1e-4 and abs(float(again) - 1.0) < 1e-5


@pytest.mark.gpu
def test_what_a_call_writes_is_not_shared_with_a_lazy_copy():
    """torch's lazy copies share memory until one of them is written."""
    from elysium_wan_amd import optim

    g = torch.Generator(device="cuda").manual_seed(3)
    grad = torch.randn(300, generator=g, device="cuda")
    p = torch.zeros(300, device="cuda")
    first, p.grad = grad.clone(), torch._lazy_clone(grad)
    optim.clip_grad_norm_([p], 0.5)
    assert torch.equal(grad, first) and not torch.equal(p.grad, first)

    got = []
    for lazy in (False, True):
        q = torch.ones(300, device="cuda", requires_grad=True)
        opt = optim.FusedAdamW([q], lr=1e-3, working_copy=True)
        opt.step(grads=[grad])
        tensors = [q.detach(), opt.state[0]["exp_avg"], opt.state[0]["exp_avg_sq"], opt.working_copies[0]]
        if lazy:
            kept = [t.clone() for t in tensors]
            shared = [torch._lazy_clone(t) for t in tensors]
            q.data = torch._lazy_clone(shared[0])
            opt._st[0]["exp_avg"], opt._st[0]["exp_avg_sq"] = torch._lazy_clone(shared[1]), torch._lazy_clone(shared[2])
            opt.working_copies[0] = torch._lazy_clone(shared[3])
        opt.step(grads=[grad])
        got.append([q.detach(), opt.state[0]["exp_avg"], opt.state[0]["exp_avg_sq"], opt.working_copies[0]])
    assert all(torch.equal(a, b) for a, b in zip(*got))
    assert all(torch.equal(a, b) for a, b in zip(kept, shared))


@pytest.mark.gpu
def test_the_step_keeps_its_tensors_until_it_is_queued():
    """The caller's lists emptied in the middle of the call, and their memory
    asked for again at once."""
    from elysium_wan_amd import optim

    g = torch.Generator(device="cuda").manual_seed(5)
    grads, accs = ([torch.randn(70001, generator=g, device="cuda") for _ in range(3)] for _ in range(2))
    got = []
    for emptied in (False, True):
        ps = [torch.ones(70001, device="cuda", requires_grad=True) for _ in grads]
        opt = optim.FusedAdamW(ps, lr=1e-3, max_norm=1.0)
        opt.step(grads=grads)
        gl, al, junk, consts = [t.clone() for t in grads], [t.clone() for t in accs], [], opt._consts

        def in_the_middle(*args):
            gl[:], al[:] = [None] * 3, [None] * 3
            junk.extend(torch.full((70001,), 1e6, device="cuda") for _ in range(12))
            return consts(*args)

        if emptied:
            opt._consts = in_the_middle
        opt.step(grads=gl, acc=al)
        assert len(junk) == 12 * emptied
        got.append([t for i, p in enumerate(ps) for t in (p.detach(), opt.state[i]["exp_avg"], opt.state[i]["exp_avg_sq"])] + [opt.grad_norm()])
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.gpu
def test_the_clip_keeps_its_gradients_until_it_is_queued():
    """The clip of a long list waits for a slot of the upload ring, the
    interpreter lock released, while another thread clears the gradients and
    asks for their memory again."""
    from elysium_wan_amd import optim

    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    torch.cuda._sleep(1000)
    start.record()
    torch.cuda._sleep(1_000_000)
    end.record()
    end.synchronize()
    busy = int(1_000_000 * 400 / max(start.elapsed_time(end), 1e-2))  # 0.4 s

    def params(value):
        ps = [torch.zeros(5000, device="cuda") for _ in range(60)]
        for p in ps:
            p.grad = torch.full((5000,), value, device="cuda")
        return ps

    ps, others = params(3.0), params(1.0)
    optim.clip_grad_norm_(others, 1e9)
    torch.cuda.synchronize()
    go, junk, cleared = threading.Event(), [], []

    def clear():
        go.wait(30)
        time.sleep(0.05)
        for p in ps:
            p.grad = None
        junk.extend(torch.full((5000,), 7.0, device="cuda") for _ in range(120))
        cleared.append(time.monotonic())

    t = threading.Thread(target=clear)
    t.start()
    torch.cuda._sleep(busy)
    for _ in range(8):  # every slot of the ring behind the busy stream
        optim.clip_grad_norm_(others, 1e9)
    go.set()
    total = optim.clip_grad_norm_(ps, 1.0)
    done = time.monotonic()
    t.join()
    torch.cuda.synchronize()
    assert cleared[0] < done, "the gradients were to be cleared during the call"
    assert abs(float(total) - 3.0 * (60 * 5000) ** 0.5) < 1e-2
    assert all(bool((j == 7.0).all()) for j in junk)


@pytest.mark.gpu
def test_a_workspace_grows_while_another_thread_asks_for_one():
    """The allocator may run Python, here a memory trace that waits for a
    second thread's call: that call must not wait for the first one's.  In a
    process of its own, for the trace stays on."""
    r = subprocess.run([sys.executable, "-u", "-c", """
import threading, torch
from torch.cuda import _gpu_trace
from elysium_wan_amd import _lib

N = _lib.load_native()
N.workspace(0, 1)
inside, done, waited = threading.Event(), threading.Event(), []

def traced(ptr):
    if not inside.is_set():
        inside.set()
        waited.append(done.wait(20))

def second():
    inside.wait(20)
    N.workspace(0, 1)
    done.set()

_gpu_trace.register_callback_for_memory_allocation(traced)
torch._C._activate_gpu_trace()
t = threading.Thread(target=second)
t.start()
grown = N.workspace(0, 8 << 20)
t.join()
assert waited == [True] and grown.numel() >= 8 << 20 and N.workspace(0, 1).data_ptr() == grown.data_ptr()
"""], cwd=ROOT, capture_output=True, text=True, timeout=90)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
def test_kernels_of_a_library_rebuilt_after_the_import_run(tmp_path):
    _copy_of_the_package(tmp_path, *LIBRARIES)
    _run(tmp_path, REPLACE + f"""
import torch
from elysium_wan_amd import _lib, fp8, optim
for name in {LIBRARIES}:
    replaced(name, os.path.join({PACKAGE!r}, name))
x = torch.randn(64, 512, device="cuda").bfloat16()
q, k = fp8.quantize(x)
assert torch.equal(fp8.dequantize(q, k, torch.bfloat16), fp8.roundtrip(x))
assert torch.equal(q.view(torch.uint8), (x * torch.exp2(-k.float()).bfloat16()).to(q.dtype).view(torch.uint8))
p = torch.zeros(300, device="cuda")
p.grad = torch.full((300,), 2.0, device="cuda")
assert abs(float(optim.clip_grad_norm_([p], 1.0)) - 2.0 * 300**0.5) < 1e-4
for name in {LIBRARIES}:
    assert str(os.stat("elysium_wan_amd/" + name).st_ino) in mapped(name), name
""")
