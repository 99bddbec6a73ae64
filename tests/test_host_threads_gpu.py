"""The native host module lets other Python threads run while it is inside the kernels' library (a launch waits there when
the device's queue is full).  A second copy of the module is bound to a library whose entry points sleep."""
import ctypes
import importlib.util
import shutil
import subprocess
import threading
import time

import pytest
import torch

from hqekv_amd import synth

pytestmark = pytest.mark.gpu
MS = 200


@pytest.fixture(scope="module")
def sleepy(tmp_path_factory):
    """-> (the module, its number of sleeps so far)"""
    from hqekv_amd import _lib
    d = tmp_path_factory.mktemp("host")
    src = ['#include <unistd.h>', 'static int calls;', 'extern "C" int sleepy_calls() { return calls; }']
    for name in _lib.EXPORTS:
        if name.endswith("_bytes"):
            src.append(f'extern "C" long {name}() {{ return 4096; }}')
        elif name == "hqekv_last_error":   # (never asked for: every call succeeds)
            src.append(f'extern "C" const char *{name}() {{ return ""; }}')
        else:
            src.append(f'extern "C" int {name}() {{ ++calls; usleep({1000 * MS}); return 0; }}')
    (d / "s.cpp").write_text("\n".join(src))
    subprocess.run(["g++", "-shared", "-fPIC", str(d / "s.cpp"), "-o", str(d / "libsleepy.so")], check=True)
    shutil.copy(_lib._PKG / "_host.so", d / "_host.so")   # (a copy has an entry table of its own)
    spec = importlib.util.spec_from_file_location("_host", d / "_host.so")
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    m.bind(str(d / "libsleepy.so"))
    return m, ctypes.CDLL(str(d / "libsleepy.so")).sleepy_calls


def _others_run(sleepy, call):
    """Does another thread make progress during every sleep of ``call``?"""
    m, calls = sleepy
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.005)
    t = threading.Thread(target=tick)
    n = calls()
    t.start()
    begin = time.perf_counter()
    assert call(m) is not None
    end = time.perf_counter()
    stop.set()
    t.join()
    slept = calls() - n
    assert slept >= 1 and end - begin >= slept * MS / 1000
    seen = [begin] + [x for x in ticks if begin < x < end] + [end]
    assert max(b - a for a, b in zip(seen, seen[1:])) < MS / 2000, "another thread stood still"


def test_decode_and_reconstruct(dev, sleepy):
    from hqekv_amd.attention import idx_cover_once
    from hqekv_amd.pack_unpack import uniform_group_quantize_pack_last_dim
    q, K, V = synth.make_qkv(1, 8, 2, 512 + 3, 128, 1, dev)
    pkv = synth.build_cache(K, V, synth.split_blocks(512, (.2, .2, .3, .3, 0), 1), 3, uniform_group_quantize_pack_last_dim)
    assert idx_cover_once([pkv[i] for i in (1, 5, 13, 21)], 512) and idx_cover_once([pkv[i] for i in (3, 9, 17, 25)], 512)
    _others_run(sleepy, lambda m: m.decode(q, pkv, True, idx_cover_once))
    _others_run(sleepy, lambda m: m.reconstruct(pkv, True, idx_cover_once))


def test_quantise_and_prompt(dev, sleepy):
    x = torch.zeros(1, 2, 64, 128, dtype=torch.float16, device=dev)
    code = torch.empty(1, 2, 64, 16, dtype=torch.int32, device=dev)
    scale = torch.empty(1, 2, 64, 4, dtype=torch.float16, device=dev)
    _others_run(sleepy, lambda m: m.quantize_into(x, 4, code, scale, scale.clone()))
    _others_run(sleepy, lambda m: m.prompt_attention(x, x, x, 0.1, True))
    _others_run(sleepy, lambda m: m.prompt_last_rows(x, x, 0.1, 20))
    _others_run(sleepy, lambda m: m.importance(torch.zeros(20, 256, dtype=torch.float16, device=dev), 128, 128))


def test_layer_steps(dev, sleepy):
    m, _ = sleepy
    q, k, v = (torch.zeros(1, h, 1, 128, dtype=torch.float16, device=dev) for h in (8, 2, 2))
    buf = torch.zeros(1, 2, 64, 128, dtype=torch.float16, device=dev)
    tables = m.StepTables(0, 0, 0, 0)
    _others_run(sleepy, lambda m: tables.step(q, k, v, (None,) * 42, buf, buf.clone(), 5, 6, None, 0, 6))
    st = m.KiviState()
    st.kt, st.vt = buf[:, :, :32].clone(), buf
    st.vcode = torch.zeros(1, 2, 64, 8, dtype=torch.int32, device=dev)
    st.vscale = torch.zeros(1, 2, 64, 4, dtype=torch.float16, device=dev)
    st.vzero = st.vscale.clone()
    st.nk = st.nv = 5
    _others_run(sleepy, lambda m: st.step(q, k, v, 6, 2, 2))


def test_compression(dev, sleepy):
    import weakref
    from hqekv_amd.cache_policy import _new_array
    x = torch.zeros(1, 2, 64 + 3, 128, dtype=torch.float16, device=dev)
    f16 = torch.zeros(64, dtype=torch.float16, device=dev)
    n = torch.tensor([64, 0, 0, 0, 0, 0])
    ring = torch.zeros(20, 96, dtype=torch.float16, device=dev)
    pkv = (None,) * 39 + (x, x.clone(), 67)
    _others_run(sleepy, lambda m: m.compress(pkv, 0, 64, f16[:2], f16, True, None, n, n.clone(), False, ring, None, _new_array, weakref.ref))
    _others_run(sleepy, lambda m: m.compress(pkv, 0, 64, f16[:2], f16, True, f16, n, n.clone(), False, ring, None, _new_array, weakref.ref))


def test_threads_with_layers_and_streams_of_their_own(dev):
    """Prompt, compressions and steps of both layers in four threads at a time: the bits of one thread after the other."""
    from hqekv_amd.decode_layer import HqeAttentionLayer
    from hqekv_amd.kivi_layer import KiviAttentionLayer
    T, steps = 200, 40

    def inputs(seed):
        g = torch.Generator().manual_seed(seed)
        return [[torch.randn(1, h, T if s == 0 else 1, 128, generator=g).half().to(dev) for h in (32, 8, 8)] for s in range(steps + 1)]
    data = [inputs(seed) for seed in range(4)]
    torch.cuda.synchronize()

    def generate(i, out):
        with torch.cuda.stream(torch.cuda.Stream()):
            hqe, kivi = HqeAttentionLayer(128, 0.2, 0.3, 0.5), KiviAttentionLayer(128, 2, 2, 32, 32)
            hqe.set_max_length(T + steps)
            a = b = None
            outs = []
            for q, k, v in data[i]:
                oa, wa, a, _ = hqe(q, k, v, None, a)
                ob, wb, b = kivi(q, k, v, None, b)
                outs += [oa, wa, ob] + ([wb] if wb is not None else [])
            torch.cuda.current_stream().synchronize()
            out[i] = [x.cpu() for x in outs + [x for x in a + b if torch.is_tensor(x)]]
    alone, together = {}, {}
    for i in range(4):
        generate(i, alone)
    threads = [threading.Thread(target=generate, args=(i, together)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(4):
        assert len(alone[i]) == len(together[i])
        for x, y in zip(alone[i], together[i]):
            assert torch.equal(x, y)
