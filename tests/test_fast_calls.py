"""The native calls behind the Python face (csrc/fast_calls.c): they make the call when every
argument is plainly right, and otherwise answer None with no exception set, so that the Python
checks decide. They are optional, in the build and in the package."""
import os
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DEV = "cuda:0"


def half(n, device="cpu"):
    return torch.zeros(n, dtype=torch.float16, device=device)


CPU_CALLS = {
    "rmsnorm": lambda h: (h(32), h(16), h(32), 2, 16, 1e-5, 0),
    "add_rmsnorm": lambda h: (h(32), h(32), h(16), h(32), 2, 16, 1e-5, 0),
    "residual_add": lambda h: (h(32), h(32), h(32), 32, 0),
    "swiglu": lambda h: (h(32), h(32), h(32), 32, 0),
    "swiglu_rows": lambda h: (h(64), h(32), 2, 16, 0),
    "linear": lambda h: (1, h(32), h(64), h(8), 2, 16, 4, 0),
    "linear_rows_residual": lambda h: (h(1024), h(2048), h(8), 2, 512, 4, 0),
    "linear_rows_swiglu": lambda h: (h(1024), h(512), 1e-5, h(4096), h(8), 2, 512, 4, 0),
    "attention_decode_fast": lambda h: (h(256), h(1024), h(1024), torch.zeros(1, dtype=torch.int32),
                                        torch.zeros(1, dtype=torch.int32), h(256),
                                        torch.zeros(1024), 1, 1, 16, 4, 1, 64, 2, 0),
}


@pytest.mark.parametrize("name", CPU_CALLS)
def test_no_answer_for_anything_but_cuda_tensors(llmk, name):
    f = getattr(llmk._fast, name)
    args = CPU_CALLS[name](half)
    assert f(*args) is None  # CPU tensors
    assert f(*args[:-1]) is None and f(*args, 0) is None  # too few and too many arguments
    for i in range(len(args)):
        for bad in (None, "x", -1, 1 << 70, 1.5, object()):
            assert f(*args[:i], bad, *args[i + 1:]) is None


def test_package_loads_without_the_native_calls(tmp_path):
    pkg = os.path.join(ROOT, "cuda-llm-engine_amd")
    for name in os.listdir(pkg):
        if not name.startswith(("_fast_calls", "__pycache__")):
            os.symlink(os.path.join(pkg, name), tmp_path / name)
    code = f"""
import importlib.util, sys, torch
spec = importlib.util.spec_from_file_location(
    "llmk", {str(tmp_path / "__init__.py")!r}, submodule_search_locations=[{str(tmp_path)!r}])
llmk = sys.modules["llmk"] = importlib.util.module_from_spec(spec)
spec.loader.exec_module(llmk)
x = torch.zeros(32, dtype=torch.float16)
try:
    llmk.residual_add(x, x, x, 32)
except llmk.LlmkError as e:
    assert "must be a CUDA tensor" in str(e)
    print("refused", llmk.version())
"""
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.startswith("refused"), out.stderr


def test_library_configures_without_python_headers(tmp_path):
    out = subprocess.run(["cmake", "-S", ROOT, "-B", str(tmp_path), "-DLLMK_BUILD_TESTS=OFF",
                          "-DCMAKE_DISABLE_FIND_PACKAGE_Python3=ON"],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    assert "without the Python face's native calls" in out.stdout


@pytest.mark.gpu
def test_operators_without_the_native_calls(llmk, monkeypatch):
    monkeypatch.setattr(llmk, "_fast", llmk._NoFastCalls())
    x = torch.randn(4, 2048, device=DEV).half()
    out = torch.empty_like(x)
    llmk.residual_add(x, x, out, x.numel())
    torch.cuda.synchronize()
    assert torch.equal(out, x + x)


@pytest.mark.gpu
def test_calls_are_made_on_the_current_stream_or_left_to_the_checks(llmk):
    x, w = torch.randn(4, 2048, device=DEV).half(), torch.ones(2048, device=DEV).half()
    out = torch.full_like(x, float("nan"))
    f = llmk._fast.rmsnorm
    ref = torch.empty_like(x)
    assert llmk.lib().llmk_rmsnorm(x.data_ptr(), w.data_ptr(), ref.data_ptr(), 4, 2048, 1e-5,
                                   torch.cuda.current_stream().cuda_stream) == 0
    assert f(x, w, out, 4, 2048, 1e-5, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        out.fill_(float("nan"))
        assert f(x, w, out, 4, 2048, 1e-5, None) == 0
        s.synchronize()
        assert torch.equal(out, ref)
    assert f(x, w, out, 4, 2048, 1e-5, s.cuda_stream) == 0
    # what the Python checks accept by another route, refuse, or name
    assert f(x, w, out, 4, 2048, 1e-5, s) is None
    assert f(torch.nn.Parameter(x), w, out, 4, 2048, 1e-5, None) is None
    assert f(x.float(), w, out, 4, 2048, 1e-5, None) is None
    assert f(x.t(), w, out, 4, 2048, 1e-5, None) is None
    assert f(x[:1], w, out, 4, 2048, 1e-5, None) is None
    assert f(x, w, out, 4, 2048, 1, None) is None
    # the library's own refusals come back as its status
    assert f(x, w, out, 4, 2044, 1e-5, None) == llmk.LLMK_ERR_SHAPE
    with pytest.raises(llmk.LlmkError):
        llmk.rmsnorm(x, w, out, 4, 2044, 1e-5)
    with pytest.raises(llmk.LlmkError, match="must be torch.float16"):
        llmk.rmsnorm(x.float(), w, out, 4, 2048, 1e-5)
    torch.cuda.synchronize()
