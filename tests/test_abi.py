"""CPU checks of the C-ABI library: it loads, exports every symbol that
include/qwen_kernels.h declares, binds like the reference engine, and its
host-side logic (sizes, synthetic generators, failure reporting) behaves.
No GPU compute is called here."""
import ctypes
import re
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
HEADER = ROOT / "include" / "qwen_kernels.h"
LIB = ROOT / "qwen35-ax7020-edge-llm_amd" / "libqwen_kernels.so"
SAMPLING_HEADER = ROOT / "include" / "qwen_sampling.h"
SAMPLING_LIB = ROOT / "qwen35-ax7020-edge-llm_amd" / "libqwen_sampling.so"


def declared_functions(header=HEADER):
    text = re.sub(r"/\*.*?\*/", "", header.read_text(), flags=re.S)
    text = "\n".join(l for l in text.splitlines() if not l.lstrip().startswith("#"))
    names = re.findall(r"(?:^|;|\})\s*(?:const\s+)?[A-Za-z_][\w]*\s*\**\s*\b([a-z_][a-z0-9_]*)\s*\(", text, re.M)
    return sorted(set(names) - {"struct", "typedef", "void"})  # "typedef void (*cb)(...)"


def exported_symbols(lib=LIB):
    out = subprocess.run(["nm", "-D", "--defined-only", str(lib)], capture_output=True, text=True, check=True)
    return {l.split()[-1] for l in out.stdout.splitlines() if " T " in l}


def test_library_built_and_loads():
    assert LIB.exists(), "run qwen35-ax7020-edge-llm_amd/build_lib.py"
    ctypes.CDLL(str(LIB))


def test_exports_every_declared_symbol():
    decl = declared_functions()
    assert len(decl) >= 40 and "bfp8_gemv" in decl and "lm_head_argmax" in decl and "bfp8_plan_create" in decl
    missing = set(decl) - exported_symbols()
    assert not missing, missing


def test_exports_nothing_undeclared():
    extra = exported_symbols() - set(declared_functions())
    assert not extra, extra


def test_sampling_library_exports_exactly_the_reference_pair():
    """libqwen_sampling.so stands in for the reference's sampling library
    (04/chat_v3.py:145-159 binds lm_head_topk and sample_from_topk)."""
    decl = set(declared_functions(SAMPLING_HEADER))
    assert decl == {"lm_head_topk", "sample_from_topk"}
    assert exported_symbols(SAMPLING_LIB) == decl
    ctypes.CDLL(str(SAMPLING_LIB))  # finds libqwen_kernels.so next to it


def test_reference_symbol_signatures_bind_like_the_engine():
    import qwen_kernels_gpu as qk

    lib = qk.load()
    # 04/qwen_real_engine.py:680-685 / :864-866
    assert lib.bfp8_gemv.argtypes == [ctypes.c_void_p] * 4 + [ctypes.c_int] * 2
    assert lib.qwen_prof_count() == 15
    names = [lib.qwen_prof_name(i).decode() for i in range(15)]
    assert names[0] == "bfp8_gemv" and names[1] == "lm_head_argmax" and names[-1] == "forward_token_c"
    assert lib.qwen_prof_name(99) == b"?" and lib.qwen_prof_get(-1) == 0.0


def test_layout_sizes():
    import qwen_kernels_gpu as qk

    lib = qk.load()
    # 3584 rows -> 56 tiles of 64; 16 blocks -> 4 exponent groups
    assert lib.bfp8_dev_mant_bytes(3584, 1024) == 3584 * 1024
    assert lib.bfp8_dev_exps_bytes(3584, 1024) == 56 * 4 * 256
    assert lib.bfp8_dev_mant_bytes(65, 128) == 2 * 64 * 128  # padded to whole tiles
    assert lib.bfp8_dev_exps_bytes(1024, 3584) == 16 * 14 * 256
    assert lib.bfp8_dev_xsplit_bytes(3584) == 56 * 128
    assert lib.bfp8_dev_mant_bytes(0, 1024) == 0 and lib.bfp8_dev_xsplit_bytes(63) == 0


def _splitmix(seed, idx):
    m = (1 << 64) - 1
    z = (seed + (idx + 1) * 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def test_synthetic_planes_follow_the_documented_hash():
    import qwen_kernels_gpu as qk

    mant, exps = qk.synth_planes(3, 128, 12345, 124, 130)
    flat = mant.reshape(-1)
    for i in (0, 1, 77, 383):
        assert flat[i] == (_splitmix(12345, i) >> 32) % 255 - 127
    ef = exps.reshape(-1)
    for i in range(ef.size):
        assert ef[i] == 124 + (_splitmix(12345 ^ 0xE7E7E7E7E7E7E7E7, i) >> 32) % 7
    assert mant.min() >= -127 and mant.max() <= 127


def test_synthetic_activation_statistics():
    import qwen_kernels_gpu as qk

    x = qk.synth_normal(200000, 9)
    assert abs(float(x.mean())) < 0.01 and abs(float(x.std()) - 1) < 0.01
    s = qk.synth_swiglu(100000, 9, 0.01, 20.0)
    frac = float(np.mean(np.abs(s) == 20.0))
    assert 0.008 < frac < 0.012
    assert np.array_equal(qk.synth_normal(64, 5), qk.synth_normal(64, 5))


@pytest.mark.parametrize("tiles,K,B,name", [
    (1, 64, 1, "rt_rows_gemv_kernel"), (385, 1024, 1, "bfp8_gemv_kernel"),
    (256, 512, 2, "span"), (257, 512, 2, "dot"), (768, 512, 2, "dot"), (769, 512, 2, "cu"), (1025, 512, 2, "dot"),
    (128, 256, 3, "span"), (129, 256, 3, "mfma"), (256, 320, 4, "span"), (512, 320, 4, "mfma"), (513, 320, 4, "cu"),
    (129, 128, 4, "dot"), (479, 768, 4, "span"), (480, 768, 4, "cu"), (543, 1024, 4, "span"), (544, 1024, 4, "cu"),
    (1025, 1024, 2, "dot"), (1600, 1024, 2, "cu"), (438, 1088, 2, "span"), (439, 1088, 2, "dot"), (439, 1088, 4, "mfma"),
    (100000, 2048, 4, "span"), (128, 768, 8, "span"), (129, 768, 8, "mfma"), (256, 1024, 8, "span"), (257, 768, 8, "cu"),
    (340, 1088, 5, "span"), (341, 1088, 5, "mfma"), (900, 2048, 8, "span"), (901, 2048, 8, "mfma"),
    (320, 3584, 8, "span"), (321, 3584, 8, "mfma"), (64, 1024, 16, "span"), (65, 1024, 16, "mfma"),
    (512, 1024, 16, "mfma"), (513, 1024, 16, "cu"), (1024, 1024, 16, "cu"), (1025, 1024, 16, "mfma"), (1281, 1024, 16, "cu"),
    (128, 1088, 16, "span"), (129, 1088, 16, "mfma"), (128, 4096, 16, "span"), (129, 4096, 16, "mfma"),
    (208, 4096, 9, "span"), (209, 4096, 9, "mfma"),
    (1, 63, 4, ""), (1, 4097, 4, ""), (1, 64, 17, ""), (0, 64, 4, "")])
def test_batch_kernel_names(tiles, K, B, name):
    """The batched GEMV's forms on both sides of the lines between them."""
    import qwen_kernels_gpu as qk

    if name in ("span", "cu", "mfma", "dot"):
        name = f"bfp8_gemv_batch_{name}_kernel"
    for M in {64 * tiles, max(64 * tiles - 63, 0)}:
        assert qk.load().bfp8_dev_gemv_batch_kernel_name(M, K, B).decode() == name


def test_device_call_without_gpu_reports_error():
    """On a host without a GPU the int entry points return an error code with
    a message; nothing falls back to the CPU."""
    import torch

    if torch.cuda.is_available():
        pytest.skip("a GPU is visible")
    import qwen_kernels_gpu as qk

    lib = qk.load()
    x = np.zeros(64, np.float32)
    out = np.zeros(64, np.float32)
    rc = lib.bfp8_dev_quantize(None, out.ctypes.data, out.ctypes.data, x.ctypes.data, 64, None)
    assert rc == qk.BFP8_EHIP
    assert b"no HIP device" in lib.bfp8_last_error()
    assert lib.bfp8_lm_head_topk(x.ctypes.data, x.ctypes.data, x.ctypes.data, 64, 64, 0, x.ctypes.data,
                                 x.ctypes.data) == 0  # invalid k: rejected before any GPU work


def test_init_without_gpu_returns_and_reports_not_ready():
    """init_kernels() cannot fail in the reference (04/qwen_kernels_opt.c:128-135)
    and the engine calls it inside its library-selection try block: without a
    GPU it returns, and bfp8_gpu_ready() says 0 with the reason."""
    import torch

    if torch.cuda.is_available():
        pytest.skip("a GPU is visible")
    code = (
        "import sys; sys.path.insert(0, %r)\n"
        "import qwen_kernels_gpu as qk\n"
        "k = qk.load(); k.init_kernels(); k.init_kernels()\n"
        "print('READY', k.bfp8_gpu_ready(), k.bfp8_last_error().decode())\n" % str(ROOT / "qwen35-ax7020-edge-llm_amd"))
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120,
                         env={"HIP_VISIBLE_DEVICES": "", "PATH": "/usr/bin:/bin"})
    assert res.returncode == 0, res.stderr
    assert "READY 0 no HIP device" in res.stdout
    assert "GPU path unavailable" in res.stderr


def test_engine_style_loader_keeps_its_numpy_path_without_gpu():
    """The engine's loader (04/qwen_real_engine.py:656-671) with the one added
    readiness check shown in INTEGRATION.md: without a GPU it ends with no
    kernel library, i.e. on the engine's own numpy path, instead of a process
    abort at the first GEMV."""
    import torch

    if torch.cuda.is_available():
        pytest.skip("a GPU is visible")
    lib = ROOT / "qwen35-ax7020-edge-llm_amd" / "libqwen_kernels.so"
    code = (
        "import ctypes\n"
        "kernels = None\n"
        "for cand in [%r]:\n"
        "    try:\n"
        "        kernels = ctypes.CDLL(cand)\n"
        "        if hasattr(kernels, 'init_kernels'):\n"
        "            kernels.init_kernels()\n"
        "        if hasattr(kernels, 'bfp8_gpu_ready') and not kernels.bfp8_gpu_ready():\n"
        "            raise OSError('GPU path unavailable')\n"
        "        break\n"
        "    except Exception:\n"
        "        kernels = None\n"
        "print('KERNELS', kernels)\n" % str(lib))
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120,
                         env={"HIP_VISIBLE_DEVICES": "", "PATH": "/usr/bin:/bin"})
    assert res.returncode == 0, res.stderr
    assert "KERNELS None" in res.stdout


def test_void_entry_point_fails_loudly_without_gpu():
    """bfp8_gemv has no error channel (04/qwen_kernels_opt.c:207): without a GPU
    the library aborts with a message instead of computing on the CPU."""
    import torch

    if torch.cuda.is_available():
        pytest.skip("a GPU is visible")
    code = (
        "import sys, numpy as np; sys.path.insert(0, %r)\n"
        "import qwen_kernels_gpu as qk\n"
        "k = qk.load(); y = np.zeros(2, np.float32); x = np.ones(64, np.float32)\n"
        "m = np.ones((2, 64), np.int8); e = np.full((2, 1), 134, np.uint8)\n"
        "k.bfp8_gemv(y.ctypes.data, x.ctypes.data, m.ctypes.data, e.ctypes.data, 2, 64)\n"
        "print('RETURNED', y)\n" % str(ROOT / "qwen35-ax7020-edge-llm_amd"))
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120,
                         env={"HIP_VISIBLE_DEVICES": "", "PATH": "/usr/bin:/bin"})
    assert res.returncode != 0 and "RETURNED" not in res.stdout
    assert "no CPU fallback" in res.stderr
