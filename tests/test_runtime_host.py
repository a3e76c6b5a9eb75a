"""The host side of the library on a CPU: gq_runtime.hip linked with
tests/native/fake_device.cpp, which stands for the HIP runtime and the kernel
launchers.  It gives device memory a size, refuses allocations on request, and
follows what the launchers are handed: that workspaces are alive and large
enough, and that the K-part sums one launch leaves reach the launch that adds
them.  What the kernels compute is not part of it."""
import ctypes as C
import dataclasses
import os
import shutil
import subprocess

import numpy as np
import pytest

import guanaco_amd.hip as H
from guanaco_amd import spec as S

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
GB = 1 << 30
SMALL = S.ModelSpec("host-test", n_layers=4, hidden=512, ff=1024, n_heads=8, n_kv_heads=2, vocab=1000,
                    layer_dtypes={k: S.Q8_0 for k in S.LAYER_WEIGHTS}, embed_dtype=S.Q8_0, lm_head_dtype=S.Q8_0)


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("fake")
    flags = ["--offload-arch=gfx950", "--offload-host-only", "-O1", "-fPIC", "-std=c++17", "-I",
             os.path.join(ROOT, "guanaco_amd", "csrc")]
    objs = []
    for src in (os.path.join(ROOT, "guanaco_amd", "csrc", "gq_runtime.hip"),
                os.path.join(ROOT, "tests", "native", "fake_device.cpp")):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        subprocess.run([HIPCC, *flags, "-x", "hip", "-c", src, "-o", objs[-1]], check=True)
    # the device code that the host object registers is not there
    nm = subprocess.run(["nm", "-u", objs[0]], capture_output=True, text=True, check=True).stdout
    fat = [w for w in nm.split() if w.startswith("__hip_fatbin")]
    stub = d / "fatbin.c"
    stub.write_text("".join(f"char {w}[64];\n" for w in fat))
    so = str(d / "libfake.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-o", so, *objs, "-x", "c++", str(stub)], check=True)
    lib = C.CDLL(so)
    for n in (n for n in H.EXPORTS if hasattr(lib, n)):
        f, g = getattr(lib, n), getattr(H.lib, n)
        f.restype, f.argtypes = g.restype, g.argtypes
    lib.fake_errors.restype = C.c_char_p
    lib.fake_count.restype, lib.fake_count.argtypes = C.c_long, [C.c_char_p]
    lib.fake_used.restype = C.c_size_t
    lib.fake_refuse_after.argtypes = [C.c_long]
    lib.fake_reset.argtypes = lib.fake_refuse_from.argtypes = [C.c_size_t]
    return lib


@pytest.fixture
def dev(built, monkeypatch):
    """The fake library in place of the real one, 288 GB free; no launch may
    have been handed dead memory or lost sums by the end."""
    built.fake_reset(288 * GB)
    monkeypatch.setattr(H, "lib", built)
    built.n = lambda what: built.fake_count(what.encode())
    yield built
    assert built.fake_errors() == b""


def prompt(dm, T, pos=0):
    return dm.prefill(np.arange(T) % 1000, pos)[0]


@pytest.mark.parametrize("T", [40, 100, 300])
@pytest.mark.parametrize("room", ["all", "o_down", "none"])
def test_prompt_sums_survive_short_workspaces(dev, T, room):
    """K-part sums of one layer's down projection are still owed when the next
    layer starts.  Where the card has room for the workspace of o and down but
    not for the larger one of q/k/v (or for none), no request of that next
    layer may free or replace it before they are added."""
    kvd, hid = SMALL.n_kv_heads * SMALL.head_dim, SMALL.hidden
    tokens = 8 * T if T <= 64 else 4 * T
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 512)
        first = prompt(dm, 2)  # the activations of up to 512 tokens are there
        if room != "all":
            assert 4 * tokens * hid < 4 * tokens * (hid + 2 * kvd)
            dev.fake_refuse_from(4 * tokens * ((hid + 2 * kvd) if room == "o_down" else 1))
        for _ in range(2):
            assert prompt(dm, T) == first
        assert dev.n("refused") > 0 or room == "all"


@pytest.mark.parametrize("how", ["h2d", "synth", "copy", "elsewhere"])
def test_weights_written_in_place(dev, how):
    """A bound projection's memory written in place through the context: later
    prompts do not multiply by a bf16 copy of what was there before."""
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 512)
        w = dm.weight(2, "wu")
        prompt(dm, 300)
        assert dev.n("dense") == 4 * SMALL.n_layers
        src = ctx.alloc(4096)
        if how == "h2d":  # its last block
            n = S.qbytes(w.dtype, w.rows, w.cols)
            ctx.check(dev.gq_hip_h2d(ctx.h, w.data + n - 34, np.zeros(34, np.uint8).ctypes.data, 34), "h2d")
        elif how == "synth":
            ctx.check(dev.gq_hip_synth_quant(ctx.h, w.data, w.dtype, w.rows, w.cols, 77), "synth")
        elif how == "copy":
            ctx.check(dev.gq_hip_copy_dev(ctx.h, w.data, src.ptr, 4096), "copy")
        else:
            src.upload(np.zeros(1024, np.float32))
        before = dev.n("dense_tile")
        prompt(dm, 300)
        stale = dev.n("dense") == 8 * SMALL.n_layers and dev.n("dense_tile") == before
        assert stale == (how == "elsewhere")


@pytest.mark.parametrize("what", ["pinned", "workspace"])
def test_failed_bind_leaves_no_model(dev, what):
    """A bind that fails for memory after it has begun to replace the bound
    model leaves none: the entry points say so instead of running on buffers
    that are gone."""
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 512)
        prompt(dm, 40)
        emb = ctx.alloc(S.qbytes(S.Q8_0, 2000, SMALL.hidden))
        dm.spec = dataclasses.replace(SMALL, vocab=2000)  # larger results: the pinned memory is made anew
        dm.model.vocab = 2000
        dm.model.embed = dm.model.lm_head = H.GqWeight(emb.ptr, S.Q8_0, 2000, SMALL.hidden)
        if what == "pinned":
            dev.fake_refuse_pinned(1)
        else:
            dev.fake_refuse_from(4 * SMALL.hidden)
        assert dev.gq_hip_model_bind(ctx.h, C.byref(dm.model)) == -4
        dev.fake_refuse_pinned(0)
        dev.fake_refuse_from(1 << 60)
        whole = C.c_int(9)
        assert dev.gq_hip_bound_layers(ctx.h, C.byref(whole)) == 0 and whole.value == 0
        assert dev.gq_hip_forward_token(ctx.h, 1, 0, None, None) == -1
        with pytest.raises(H.HipError, match="no model bound"):
            prompt(dm, 40)
        assert dev.gq_hip_model_bind(ctx.h, C.byref(dm.model)) == 0  # and it can be bound again
        prompt(dm, 300)
        assert dev.gq_hip_forward_token(ctx.h, 1, 300, None, None) >= 0


@pytest.mark.parametrize("what", ["device", "retry", "pinned", "bind", "upload"])
def test_refused_memory_is_no_launch_error(dev, what):
    """Launches are checked by the thread's last error: memory that was refused
    before one, and then done without or found elsewhere, is not its failure."""
    dev.fake_reset(GB)
    with H.Context(0) as ctx:
        x = ctx.alloc(4096)
        if what in ("device", "retry"):
            prompt(H.DeviceModel(ctx, SMALL, 512), 300)
            rest = GB - 256 - dev.fake_used()
            assert bool(dev.gq_hip_malloc(ctx.h, rest + (copies(SMALL) // 2 if what == "retry" else GB))) == (what == "retry")
        else:
            dev.fake_refuse_pinned(1)
            if what == "pinned":
                assert not dev.gq_hip_host_alloc_pinned(4096)
            elif what == "upload":
                assert not dev.gq_hip_upload_weight(ctx.h, np.zeros(4096, np.uint8).ctypes.data, 4096)
            else:
                with pytest.raises(H.HipError, match="pinned"):
                    H.DeviceModel(ctx, SMALL, 512)
            dev.fake_refuse_pinned(0)
        assert dev.gq_hip_copy_dev(ctx.h, x.ptr, x.ptr + 2048, 2048) == 0


def test_refused_token_log(dev):
    """A decode loop whose token log finds no memory fails, and single steps
    go on with the log that their captured graph writes."""
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 8192)
        step = lambda: dev.gq_hip_forward_token(ctx.h, 1, 0, None, None)  # noqa: E731
        assert step() == 3
        dev.fake_refuse_from(4 * 5000)
        with pytest.raises(H.HipError):
            dm.decode_loop(1, 0, 5000)
        assert step() == 3 and step() == 3
        dev.fake_refuse_from(1 << 60)
        dm.decode_loop(1, 0, 5000)
        assert step() == 3


@pytest.mark.parametrize("granted", [0, 1])
def test_refused_attention_partials(dev, granted):
    """Decode attention without a bound model grows its own partials: when one
    of the two finds no memory the call fails, and a smaller one afterwards
    has both again."""
    with H.Context(0) as ctx:
        q = ctx.alloc(4 * 8 * 64)
        ctx.kv_init(1, 2, 64, 64, 500000.0)
        assert ctx.attention_dev(0, 3, 8, q, q) == 0
        ctx.kv_init(1, 2, 64, 4096, 500000.0)
        dev.fake_refuse_after(granted)
        assert ctx.attention_dev(0, 3, 8, q, q) == -4
        dev.fake_refuse_after(-1)
        ctx.kv_init(1, 2, 64, 64, 500000.0)
        assert ctx.attention_dev(0, 3, 8, q, q) == 0


def copies(spec):
    """bytes of the bf16 copies as the stand-in lays them out"""
    per = sum(2 * np.prod(spec.shape(k)) for k in ("wq", "wk", "wv", "wo", "wd")) + 4 * np.prod(spec.shape("wg"))
    return int(per) * spec.n_layers


def test_copies_are_made_by_the_first_long_prompt(dev):
    """The bf16 copies of the weights cost time and 2 bytes a weight, so only a
    prompt that uses them makes them: not a bind, a step, a short prompt, or
    any prompt in the mode that runs token by token."""
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 4096)
        dm.forward(1, 0)
        prompt(dm, 256)
        assert dev.gq_hip_set_prefill_mode(ctx.h, 1) == 0
        prompt(dm, 600)
        assert dev.n("dense_tile") == 0
        assert dev.gq_hip_set_prefill_mode(ctx.h, 0) == 1
        used = dev.fake_used()
        prompt(dm, 257)
        made = dev.n("dense_tile")
        assert made == 6 * SMALL.n_layers and dev.fake_used() >= used + copies(SMALL)
        prompt(dm, 3000)  # once
        assert dev.n("dense_tile") == made and dev.n("dense") == 4 * SMALL.n_layers * 3


def test_copies_only_where_there_is_room(dev):
    """A card of which the copies would take a quarter or more of what is free
    runs prompts without them, and asks again once something is given back."""
    dev.fake_reset(GB)
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 512)
        prompt(dm, 200)  # the activations
        held = ctx.alloc(GB - 256 - dev.fake_used() - 4 * copies(SMALL))
        prompt(dm, 300)
        prompt(dm, 300)
        assert dev.n("dense") == dev.n("dense_tile") == 0
        held.free()
        prompt(dm, 300)
        assert dev.n("dense") == 4 * SMALL.n_layers
        # not even a layer's copy can be had: all go, and nothing is asked for
        # again until something is given back
        dev.gq_hip_model_bind(ctx.h, C.byref(dm.model))
        dev.fake_refuse_from(copies(SMALL) // SMALL.n_layers)
        prompt(dm, 300)
        n = dev.n("refused")
        prompt(dm, 300)
        assert n > 0 and dev.n("dense") == 4 * SMALL.n_layers and dev.n("refused") == n


def test_what_takes_the_copies_back(dev):
    """A request that needs their room takes the copies back; one that could
    not be met even so, or that its caller can do without (K parts, the
    attention's key parts, the sampler's lists, a longer chunk), does not."""
    dev.fake_reset(GB)
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 8192)
        x = ctx.alloc(4 * 200000)
        prompt(dm, 257)
        made = dev.n("dense_tile")
        assert made == 6 * SMALL.n_layers

        def fill(rest):
            return ctx.alloc(GB - 256 - dev.fake_used() - rest)

        def kept():
            n = dev.n("dense")
            prompt(dm, 300)
            return dev.n("dense") == n + 4 * SMALL.n_layers and dev.n("dense_tile") == made

        with pytest.raises(H.HipError):
            ctx.alloc(GB)
        assert kept()
        held = fill(1 << 20)
        n = dev.n("refused")
        chunks = dev.n("chunk")
        prompt(dm, 4000, 4000)  # two chunks of 2000, or in 512 tokens at most
        assert dev.n("refused") > n and dev.n("chunk") == chunks + 8
        n = dev.n("refused")
        assert dev.gq_hip_sample_dev(ctx.h, x.ptr, 200000, 1.0, 40, 1.0, 7) == 5
        assert dev.n("refused") > n and dev.n("topk_replay") == 1
        assert kept()
        more = ctx.alloc(copies(SMALL) // 2)  # fits where the copies were
        assert not kept() and dev.n("dense_tile") == made
        more.free()
        held.free()


def test_what_takes_the_prompt_workspaces_back(dev):
    """Between prompts their workspaces (up to 2048 tokens of activations and K
    parts) are room that a request may need: one that fits with it gets it, one
    that would not fit even so leaves them, and they go before the copies do."""
    dev.fake_reset(GB)
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 4096)
        prompt(dm, 2)
        bare = dev.fake_used()
        first = prompt(dm, 2048)
        used = dev.fake_used()
        held = used - bare - dev.gq_hip_prefill_copy_bytes(ctx.h)
        assert held > 20 << 20
        with pytest.raises(H.HipError):
            ctx.alloc(GB)
        assert dev.fake_used() == used
        room = ctx.alloc(GB - 256 - used + held // 2)
        assert dev.gq_hip_prefill_copy_bytes(ctx.h) == copies(SMALL)
        for T in (2048, 300, 40):
            assert prompt(dm, T) == first
        room.free()
        assert prompt(dm, 2048) == first
        room = ctx.alloc(GB - 256 - dev.fake_used() + held + copies(SMALL) // 2)
        assert dev.gq_hip_prefill_copy_bytes(ctx.h) == 0
        room.free()
        assert prompt(dm, 2048) == first


def test_copies_switched_off_and_on(dev):
    """gq_hip_set_prefill_copies(0) gives the copies back and makes no more; 1
    allows them again; the setting outlives a bind."""
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 512)
        for bad in (-1, 2):
            assert dev.gq_hip_set_prefill_copies(ctx.h, bad) == -1
        assert dev.gq_hip_prefill_copy_bytes(ctx.h) == 0
        prompt(dm, 300)
        assert dev.gq_hip_prefill_copy_bytes(ctx.h) == copies(SMALL)
        used = dev.fake_used()
        assert dev.gq_hip_set_prefill_copies(ctx.h, 0) == 1
        assert dev.gq_hip_prefill_copy_bytes(ctx.h) == 0 and dev.fake_used() <= used - copies(SMALL)
        n = dev.n("dense")
        prompt(dm, 300)
        dev.gq_hip_model_bind(ctx.h, C.byref(dm.model))
        prompt(dm, 300)
        assert dev.n("dense") == n
        assert dev.gq_hip_set_prefill_copies(ctx.h, 1) == 0
        prompt(dm, 300)
        assert dev.n("dense") == n + 4 * SMALL.n_layers and dev.gq_hip_prefill_copy_bytes(ctx.h) == copies(SMALL)


def test_no_copies_of_misaligned_weights(dev):
    """Weights off a 16-byte boundary have no copies, and nothing is allocated
    for them."""
    with H.Context(0) as ctx:
        dm = H.DeviceModel(ctx, SMALL, 512)
        w = dm.layers[2].wk
        room = ctx.alloc(S.qbytes(S.Q8_0, w.rows, w.cols) + 16)
        w.data = room.ptr + 4
        assert dev.gq_hip_model_bind(ctx.h, C.byref(dm.model)) == 0
        prompt(dm, 300)
        used = dev.fake_used()
        prompt(dm, 300)
        assert dev.n("dense_tile") == dev.n("dense") == 0 and dev.fake_used() == used
