"""The tracked calls of ``perf/cases.py`` at small sizes: what each call returns
lies within its stated tolerance of the file's own 64-bit restatement."""

import importlib.util
import os

import pytest
import torch

from conftest import REPO

pytestmark = pytest.mark.gpu

CASES = [("call", "plumbing", 2, 256, 64, "bf16"), ("call", "any_length", 3, 333, 64, "fp16"),
         ("call", "elementwise", 2, 1000, 128, "bf16"), ("call", "dynamic", 2, 1000, 128, "bf16"),
         ("call", "mxfp8", 2, 700, 128, "bf16"), ("call", "blasst", 2, 1500, 128, "bf16"),
         ("call", "defaults", 2, 512, 64, "fp32"), ("call", "defaults_sdpa", 2, 777, 128, "bf16"),
         ("cached", "dynamic", 2, 512, 64, "fp16"), ("prepare", "mxfp8", 3, 700, 128, "bf16"),
         ("prepare", "dynamic", 2, 512, 64, "fp32"), ("quantise", "elementwise", 2, 700, 128, "bf16"),
         ("quantise", "defaults", 2, 512, 64, "bf16"), ("simulate", "defaults", 2, 512, 128, "bf16")]


def _cases():
    spec = importlib.util.spec_from_file_location("tracked_cases", os.path.join(REPO, "perf", "cases.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _pairs(got, want, name=""):
    if isinstance(want, dict):
        assert set(got) == set(want), name
        for k in want:
            yield from _pairs(got[k], want[k], f"{name}.{k}")
    elif want is None:
        assert got is None, name
    else:
        yield name, got, want


@pytest.mark.parametrize("kind,recipe,h,n,d,dtype", CASES)
def test_call_matches_its_restatement(gpu, kind, recipe, h, n, d, dtype):
    c = _cases()
    case = dict(kind=kind, recipe=recipe, B=1, H=h, N=n, D=d, dtype=dtype)
    if recipe == "blasst":
        case["fill"] = "mean_a1.5"
    got, want, tol = c.run(c.prepare(case, 3)), c.exact(case, 3), c.tolerance(case)
    for name, a, b in _pairs(got, want):
        if not torch.is_tensor(b):
            assert a == pytest.approx(b, rel=1e-12), name
            continue
        assert a.shape == b.shape, name
        if tol == "exact" or not a.is_floating_point():
            assert torch.equal(a.double(), b.double()), name
            continue
        a, b = a.double(), b.double()
        assert float((a - b).norm()) <= tol["rel"] * float(b.norm()), name
        bound = tol["max"] * b.abs().clamp_min(float(b.pow(2).mean().sqrt()))
        assert bool(((a - b).abs() <= bound).all()), name
