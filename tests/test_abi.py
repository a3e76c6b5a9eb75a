"""The C-ABI library loads and exports every entry point include/gq_hip.h
declares; without a GPU the context factory fails cleanly (NULL), mirroring
the reference's backend factory returning NULL for an unavailable device
(backend.c:27-33, test_backend.c:92-112)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared(header):
    src = open(os.path.join(ROOT, "include", header)).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(gq_hip_\w+)\s*\(", src)))


def test_every_declared_symbol_is_exported():
    import guanaco_amd.hip as H
    lib = ctypes.CDLL(H.LIB_PATH)
    names = declared("gq_hip.h")
    assert len(names) >= 40
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing
    # and the Python mirror binds each of them
    assert sorted(H.EXPORTS) == names


def test_no_device_means_null_context():
    import guanaco_amd.hip as H
    if H.device_count() > 0:
        pytest.skip("a GPU is present")
    assert not H.lib.gq_hip_create(0)
    with pytest.raises(H.HipError):
        H.Context(0)


def test_prompt_attention_rule_for_unsupported_groups():
    """The workspace rule of the prompt attention (plain host code) for head
    geometries that no kernel takes: no rows, where it had divided by 16 / G =
    0 for more than 16 query heads per KV head and ended the process."""
    import subprocess
    import sys
    code = """
import ctypes, guanaco_amd.hip as H
f = ctypes.CDLL(H.LIB_PATH)._Z14gq_flash_partsiiiiii  # gq_flash_parts(ntok, pos, n_heads, n_kv, hd, n_cu)
f.restype = ctypes.c_size_t
for nh, nkv, hd in ((32, 1, 64), (96, 2, 128), (17, 1, 64), (16, 1, 64), (24, 8, 128), (32, 8, 96), (0, 8, 64)):
    for ntok, pos in ((1, 0), (37, 8000), (512, 3584)):
        assert f(ntok, pos, nh, nkv, hd, 256) == 0, (nh, nkv, hd)
assert f(37, 8000, 32, 8, 128, 256) > 0
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT)
    assert r.returncode == 0, (r.returncode, r.stderr[-500:])


@pytest.mark.parametrize("ntok,pos,nh,nkv,hd,split", [
    (900, 0, 8, 8, 128, 0), (768, 0, 8, 8, 128, 0), (900, 300, 8, 8, 128, 4), (768, 0, 8, 1, 128, 0), (900, 0, 8, 4, 128, 0),
    (512, 3584, 32, 8, 128, 2), (128, 2000, 32, 8, 128, 8), (37, 8000, 32, 8, 128, 8), (77, 301, 32, 4, 64, 0),
])
def test_prompt_attention_rule(ntok, pos, nh, nkv, hd, split):
    """Parts of the keys (0: one part, or the fp32 kernel) at launches that were
    timed with every choice, at 256 CUs.  The first five had gone to five or six
    parts, 1.2 to 1.25 times as slow."""
    import guanaco_amd.hip as H
    f = ctypes.CDLL(H.LIB_PATH)._Z14gq_flash_partsiiiiii  # gq_flash_parts(ntok, pos, n_heads, n_kv, hd, n_cu)
    f.restype = ctypes.c_size_t
    assert f(ntok, pos, nh, nkv, hd, 256) == split * ntok * nh


def test_reference_patch_applies_and_builds(tmp_path):
    """The drop-in as a maintainer applies it: guanaco_amd/host/reference-hip.patch
    applies to the reference's src/ tree as it is, and with hip_backend.c /
    .h added the tree compiles with -DUSE_HIP=1 (the HIP backend under
    -Wall -Wextra -Werror) into the engine library and the command-line
    program, which export the factory (backend.h:41-52) and every hook
    hip_backend.h declares."""
    import subprocess
    from oracle import ref_available
    if not ref_available():
        pytest.skip("reference sources / oracle/_ref not present")
    out = tmp_path / "ref_hip"
    r = subprocess.run(["sh", os.path.join(ROOT, "oracle", "build_ref_hip.sh"), str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    src = open(os.path.join(ROOT, "guanaco_amd", "host", "hip_backend.h")).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    names = sorted(set(re.findall(r"\b(hip_\w+|backend_hip_\w+)\s*\(", src)))
    assert {"hip_backend_upload", "hip_backend_bind_model", "hip_backend_prefill", "hip_layer_ready",
            "hip_backend_layer", "hip_backend_kv_sync", "hip_upload_weight", "hip_backend_whole",
            "hip_backend_prompt", "hip_backend_forward_sample", "hip_backend_host_kv"} <= set(names)
    lib = ctypes.CDLL(str(out / "libref_hip.so"))
    missing = [n for n in names + ["backend_create", "backend_kernels", "backend_destroy", "backend_hip_create",
                                   "forward", "transformer_layer", "gpu_prefill", "kv_cache_load"]
               if not hasattr(lib, n)]
    assert not missing, missing
    patched = {l.split()[1][2:] for l in open(os.path.join(ROOT, "guanaco_amd", "host", "reference-hip.patch"))
               if l.startswith("+++ ")}
    assert {"backend/backend.c", "backend/backend_internal.h", "include/backend.h", "include/tokenizer.h",
            "tokenizer/tokenizer.c", "main.c", "engine/loader.c", "engine/engine.c", "engine/generate.c",
            "engine/chat.c", "engine/gpu_prefill.c"} <= patched


def test_patched_cli_device_switch(tmp_path):
    """--device hip in the patched command line (tokenizer.c:337-343,
    :385-392, :420-433; main.c:14-42): an unknown kind is refused and names
    hip among the kinds; without a GPU the HIP backend request fails with a
    message instead of falling back."""
    import subprocess
    cli = os.path.join(ROOT, "oracle", "_ref", "guanaco_hip")
    if not os.path.exists(cli):
        pytest.skip("oracle/_ref/guanaco_hip not built")
    r = subprocess.run([cli, "--device", "bogus", "--model", "x"], capture_output=True, text=True, cwd=tmp_path)
    assert r.returncode == 1 and "auto|cpu|cuda|hip" in r.stderr
    import guanaco_amd.hip as H
    if H.device_count() > 0:
        pytest.skip("a GPU is present")
    r = subprocess.run([cli, "--device", "hip", "--model", str(tmp_path / "none.gguf")], capture_output=True,
                       text=True, cwd=tmp_path)
    assert "HIP backend requested but unavailable" in r.stderr
