"""Static gates on the sources (in the spirit of the reference's
scripts/static_checks.py:14-49): nothing on the product path may make a
result depend on scheduling order or on a library's choice of algorithm."""

from __future__ import annotations

import re
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "lockstep_amd" / "csrc"
PACKAGE = ROOT / "lockstep_amd"


def strip_comments(text: str) -> str:
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.sub(r"//[^\n]*", "", text)


def test_kernels_use_no_atomics_and_no_library_math():
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")):
        code = strip_comments(path.read_text())
        for banned in ("atomicAdd", "atomicMax", "atomicMin", "atomicExch", "atomicCAS", "__hip_atomic",
                       "rocblas", "hipblas", "miopen", "hipcub", "rocprim", "__shfl_down", "__reduce_"):
            assert banned not in code, f"{path.name} uses {banned}"
        assert "-ffast-math" not in code


def test_kernels_are_built_without_contraction_and_for_gfx950_only():
    from lockstep_amd.ops import build

    assert "-ffp-contract=off" in build.FLAGS and "--offload-arch=gfx950" in build.FLAGS
    assert "-packed-fp32-ops" in build.FLAGS
    assert not any("fast-math" in f for f in build.FLAGS)


def test_a_barrier_inside_a_wave_has_its_fences():
    """__builtin_amdgcn_wave_barrier orders instructions and is declared to touch no memory: where lanes of a wave hand each other
    values through LDS, it takes a release fence in front of it and an acquire fence behind it."""
    barrier = "__builtin_amdgcn_wave_barrier();"
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")):
        lines = [line.strip() for line in strip_comments(path.read_text()).splitlines() if line.strip()]
        for i, line in enumerate(lines):
            if barrier in line:
                assert lines[i - 1] == '__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");', (path.name, lines[i - 1])
                assert lines[i + 1] == '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");', (path.name, lines[i + 1])


def test_product_path_calls_no_library_model_code():
    """No torch matrix products, attention, softmax or norms in the package:
    those are the hand-written kernels' job (the sampler's float64 top-p on the
    host is the named exception, as in the reference)."""
    banned = [r"torch\.matmul", r"torch\.bmm", r"torch\.einsum", r"F\.linear", r"scaled_dot_product_attention",
              r"torch\.nn\.functional", r"torch\.softmax", r"\.softmax\(", r"F\.rms_norm", r"torch\.rms_norm", r"layer_norm\(",
              r"import transformers", r"from transformers", r"import vllm", r"@ self\.", r"\.mm\("]
    for path in sorted(PACKAGE.rglob("*.py")):
        code = path.read_text()
        for pattern in banned:
            assert not re.search(pattern, code), f"{path.relative_to(ROOT)} matches {pattern}"


def test_engine_does_not_import_tests_or_working_files():
    for path in sorted(PACKAGE.rglob("*.py")) + [ROOT / "bench.py", ROOT / "bin" / "trace_run"]:
        code = path.read_text()
        assert "_work" not in code, path
        assert not re.search(r"^\s*(from|import)\s+(tests|plain)\b", code, flags=re.M), path


def test_narrow_column_blocks_cost_the_streaming_products_no_round():
    """A round of a walk costs its barrier and its fold however narrow its block is: blocks of 12 columns only where the walks
    have no more rounds with them (the heads of 151,936 columns and the widths of three rounds and more do)."""
    import ctypes

    from lockstep_amd.ops import build

    columns = ctypes.CDLL(str(build.build_core())).ls_gemm_stream_columns
    for walkers in (128, 256, 512):
        for n in [*range(1, 20 * walkers, 7), 10240, 14336, 22016, 32000, 151936]:
            rounds = {c: -(-(-(-n // c)) // walkers) for c in (12, 16)}
            assert columns(n, walkers) == (12 if rounds[12] == rounds[16] else 16), (n, walkers)
    assert [columns(n, 256) for n in (4608, 6144, 7168, 9216, 10240, 14336, 22016, 151936)] == [12, 12, 16, 12, 16, 16, 16, 16]


def test_the_products_tile_numbering_refuses_a_band_of_no_rows():
    """A tuning macro of 0 would be a division by zero in device code."""
    import shutil
    import subprocess

    import pytest

    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).is_file():
        pytest.skip("no hipcc")
    check = [hipcc, "--offload-arch=gfx950", "--offload-host-only", "-fsyntax-only", "-std=c++17", str(CSRC / "gemm.hip")]
    assert subprocess.run(check, capture_output=True).returncode == 0
    refused = subprocess.run(check + ["-DLS_GEMM_GROUP_M=0"], capture_output=True, text=True)
    assert refused.returncode != 0 and "static assertion failed" in refused.stderr
