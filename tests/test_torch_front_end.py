"""What the torch front end's host path decides before any kernel runs: operands it refuses, plans it picks, how it is
loaded.  No GPU is needed; tensors are on the CPU, which the calls refuse last."""

import ctypes
import json
import os
import random
import subprocess
import sys
import types

import pytest
import torch
import torch.autograd.forward_ad as fwAD

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi, moe, ops, planner
from gpu_ragged_dot_amd import _native as _native_loader
from gpu_ragged_dot_amd._native import lib as _native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _routing(tokens, top_k):
    slots = torch.arange(tokens * top_k, dtype=torch.int32)
    return moe.Routing(torch.tensor([tokens * top_k], dtype=torch.int32), slots, slots, tokens, top_k)


@pytest.mark.parametrize("call", ["gmm x", "gmm A", "tgmm x", "tgmm y", "dispatch", "combine y", "combine weights"])
@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_tangents_are_refused(call, grad):
    with fwAD.dual_level():
        plain = lambda *s: torch.randn(*s)
        dual = lambda *s: fwAD.make_dual(torch.randn(*s, requires_grad=grad), torch.randn(*s))
        gs = torch.tensor([4], dtype=torch.int32)
        calls = {
            "gmm x": lambda: rd.gmm(dual(4, 8), plain(1, 8, 8), gs),
            "gmm A": lambda: rd.gmm(plain(4, 8), dual(1, 8, 8), gs),
            "tgmm x": lambda: rd.tgmm(dual(4, 8), plain(4, 8), gs),
            "tgmm y": lambda: rd.tgmm(plain(4, 8), dual(4, 8), gs),
            "dispatch": lambda: moe.dispatch(dual(4, 8), _routing(4, 1)),
            "combine y": lambda: moe.combine(dual(4, 8), _routing(4, 1)),
            "combine weights": lambda: moe.combine(plain(4, 8), _routing(4, 1), dual(4, 1)),
        }
        with pytest.raises(NotImplementedError, match="forward-mode"):
            calls[call]()


class _HiddenKernels:
    """Stands in for the native module on CPU tensors: its results are written behind torch's back, as a kernel writes them."""

    @staticmethod
    def _of(value):
        out = torch.empty_like(value, requires_grad=False)
        ctypes.memmove(out.data_ptr(), value.detach().contiguous().data_ptr(), value.numel() * value.element_size())
        return out.requires_grad_(value.requires_grad)

    def gmm(self, x, A, gs, *_):
        return self._of(x @ A[0])

    def tgmm(self, x, y, gs, *_):
        return self._of((x.t() @ y)[None])

    def moe_route(self, ids, groups):
        return tuple(self._of(ids.flatten() + i) for i in range(3))

    def moe_dispatch(self, h, *_):
        return self._of(h * 3)

    def moe_combine(self, y, weights, *_):
        return self._of(y if weights is None else y * weights)


@pytest.mark.parametrize("call", ["gmm", "tgmm", "route", "dispatch", "combine", "combine with weights"])
@pytest.mark.parametrize("grad", [False, True])
def test_traces_record_the_call_and_not_its_allocation(call, grad, monkeypatch):
    monkeypatch.setattr(ops, "_native", _HiddenKernels())
    monkeypatch.setattr(moe, "_native", _HiddenKernels())
    gs, r = torch.tensor([16], dtype=torch.int32), _routing(16, 1)
    floats = lambda *shapes: [torch.randn(*s, requires_grad=grad) for s in shapes]
    fn, inputs = {
        "gmm": (lambda x, A: rd.gmm(x, A, gs), lambda: floats((16, 24), (1, 24, 8))),
        "tgmm": (lambda x, y: rd.tgmm(x, y, gs), lambda: floats((16, 24), (16, 8))),
        "route": (lambda ids: tuple(moe.route(ids, 4)[:3]), lambda: [torch.randint(4, (16, 1), dtype=torch.int32)]),
        "dispatch": (lambda h: moe.dispatch(h, r), lambda: floats((16, 8))),
        "combine": (lambda y: moe.combine(y, r), lambda: floats((16, 8))),
        "combine with weights": (lambda y, w: moe.combine(y, r, w), lambda: floats((16, 8), (16, 1))),
    }[call]
    traced = torch.jit.trace(fn, tuple(inputs()), check_trace=False)
    for _ in range(2):  # on other inputs than the recorded ones
        args = inputs()
        got, want = traced(*args), fn(*args)
        for a, b in zip(*((t,) if isinstance(t, torch.Tensor) else t for t in (got, want))):
            assert torch.equal(a, b)


@pytest.mark.parametrize("op", ["gmm", "gmm trans_rhs", "tgmm"])
def test_explicit_blocks_plan_what_the_call_computes(op, monkeypatch):
    """One plan for a product alone, three where an operand asks for a gradient; an operand that is copied because of its
    strides does not count as one at an odd address."""
    asked, handed = [], []
    real = planner.select_plan
    monkeypatch.setattr(planner, "select_plan", lambda *a, **kw: (asked.append((a, kw)), real(*a, **kw))[1])
    native = types.SimpleNamespace(gmm=lambda *a: handed.append(a[-1]), tgmm=lambda *a: handed.append(a[-1]))
    monkeypatch.setattr(ops, "_native", native)
    gs = torch.tensor([64, 64], dtype=torch.int32)
    blocks = dict(block_m=128, block_k=128, block_n=128)
    bf16 = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    call = {"gmm": lambda x, o: rd.gmm(x, o(2, 64, 64), gs, **blocks), "gmm trans_rhs": lambda x, o: rd.gmm(x, o(2, 64, 64), gs, trans_rhs=True, **blocks),
            "tgmm": lambda x, o: rd.tgmm(x, o(128, 64), gs, **blocks)}[op]
    call(bf16(128, 64), bf16)
    call(bf16(128, 64), lambda *s: bf16(*s).requires_grad_())
    with torch.no_grad():
        call(bf16(128, 64), lambda *s: bf16(*s).requires_grad_())
    assert [len(p) for p in handed] == [1, 3, 1] and len(asked) == 5
    assert all(kw["aligned"] for _, kw in asked) and all(p[0] == handed[0][0] for p in handed)
    del asked[:], handed[:]
    call(bf16(128, 72)[:, 1:65], bf16)  # strided, at an odd element: a copy is multiplied
    call(bf16(128 * 64 + 1)[1:].view(128, 64), bf16)  # contiguous, at an odd element
    assert [kw["aligned"] for _, kw in asked] == [True, False]


def test_native_and_python_planner_agree():
    """One rule, written twice: what a torch call gets and what planner.select_plan() - the JAX front end, the benchmark and
    the tests of the rule itself - says."""
    assert planner.tuned_plans(), "the tuned table is part of the rule"
    shapes = [key for key, _ in planner.tuned_plan_fields()]
    rng = random.Random(0)
    size = lambda hi: rng.choice([round(2 ** rng.uniform(0, hi)), 8 * round(2 ** rng.uniform(0, hi - 3))])
    shapes += [(op, size(15), size(13), size(13), round(2 ** rng.uniform(0, 8))) for op in range(3) for _ in range(300)]
    for op, m, k, n, g in shapes:
        for code in range(5):
            for aligned in (True, False):
                want = ops._fields(planner.select_plan(op, m, k, n, g, dtype=code, aligned=aligned))
                assert _native.pick_plan(op, m, k, n, g, code, aligned) == want, (op, m, k, n, g, code, aligned)


def test_a_tuned_table_of_another_build_does_not_prevent_the_import(tmp_path):
    """An entry that names a tile shape this build does not have refuses its own call and no other."""
    table = {"gmm:m64:k64:n64:g2": {"variant": "no_such_shape"}, "gmm:m64:k64:n128:g2": {"variant": "t64x64x64_w2x2", "group_m": 3},
             "gmm:m64:k64:n192:g2": {}, "gmm:m64:k64:n256:g2": None, "tgmm:m64": {"variant": "t64x64x64_w2x2"}, "tuned on": "a Tuesday"}
    path = tmp_path / "plans.json"
    path.write_text(json.dumps(table))
    code = ("from gpu_ragged_dot_amd import _capi, planner\nfrom gpu_ragged_dot_amd._native import lib\n"
            "pick = lambda n: lib.pick_plan(0, 64, 64, n, 2, 0, True)\nids = range(_capi.lib.rd_num_variants())\n"
            "assert pick(64)[0] not in ids and pick(192)[0] not in ids\n"
            "assert pick(128)[:2] == (planner.variant_id('t64x64x64_w2x2'), 3)\n"
            "assert pick(256)[0] in ids and pick(320)[0] in ids\n")
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, RAGGED_DOT_TUNED_PLANS=str(path)), cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr


def test_a_torch_without_rocm_counts_as_none(tmp_path):
    """A JAX process often has a CPU build of torch installed: the library builds and the package imports beside it, without
    the torch front end."""
    code = ("import sys, torch\ntorch.version.hip = None\nimport gpu_ragged_dot_amd as rd\n"
            "from gpu_ragged_dot_amd import _capi, planner\n"
            "assert 'gpu_ragged_dot_amd._native' not in sys.modules and not hasattr(rd, 'ragged_dot')\n"
            "planner.select_plan(_capi.OP_GMM, 512, 512, 512, 4)\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    csrc = os.path.join(ROOT, "gpu_ragged_dot_amd", "csrc")
    for variables, built in (([], True), ([f"TORCH_DIR={tmp_path}"], False), (["TORCH_DIR="], False)):
        r = subprocess.run(["make", "-n", "-W", "rd_torch.cpp", "-C", csrc, *variables], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0 and ("-o _rd_torch.so" in r.stdout) == built, (variables, r.stdout, r.stderr)


def test_the_native_module_is_rebuilt_for_another_torch():
    csrc = os.path.join(ROOT, "gpu_ragged_dot_amd", "csrc")
    dry = lambda *v: subprocess.run(["make", "-n", "-C", csrc, *v, "_rd_torch.so"], capture_output=True, text=True, timeout=300)
    other = dry("TORCH_ID=torch-0.0-cpython-00")
    assert other.returncode == 0 and "-o _rd_torch.so" in other.stdout, other.stderr
    if os.path.isdir(os.path.join(csrc, "build")):  # (a tree that was shipped built has no record of what it was built with)
        assert "-o _rd_torch.so" not in dry().stdout


def test_a_module_that_does_not_fit_says_what_to_do(tmp_path, monkeypatch):
    """A module built with another torch misses symbols of this one."""
    path = tmp_path / "_rd_torch.so"
    path.write_bytes(b"\x7fELF")
    monkeypatch.setattr(_native_loader, "PATH", str(path))
    with pytest.raises(ImportError, match="build it again"):
        _native_loader._load()


@pytest.mark.parametrize("call", ["gmm", "tgmm", "tgmm columns", "route", "dispatch", "combine"])
def test_sizes_beyond_32_bits_are_refused(call):
    """The kernels take 32-bit sizes; one more than 2^32 must not pass as the 9 it is in its low half."""
    m = 2 ** 32 + 9
    wide = lambda *s: torch.zeros(1, *s[1:]).expand(*s)  # no memory behind it
    gs = torch.tensor([9], dtype=torch.int32)
    r = _routing(9, 1)._replace(tokens=m)
    calls = {"gmm": lambda: rd.gmm(wide(m, 8), torch.zeros(1, 8, 8), gs), "tgmm": lambda: rd.tgmm(wide(m, 8), wide(m, 8), gs),
             "tgmm columns": lambda: rd.tgmm(torch.zeros(9, 8), torch.zeros(9, 1).expand(9, m), gs),
             "route": lambda: moe.route(torch.zeros(1, 1, dtype=torch.int32).expand(m, 1), 4),
             "dispatch": lambda: moe.dispatch(wide(m, 8), r), "combine": lambda: moe.combine(wide(m, 8), r)}
    with pytest.raises(_capi.RaggedDotError, match="beyond"):
        calls[call]()
