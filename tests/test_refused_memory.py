"""Device memory running out, on the CPU: a stand-in for the HIP runtime
(fake_hip.c) refuses allocations of chosen sizes. A refused optional buffer must
leave the call on its other path, a refused mandatory one must fail the call, and
neither may spoil a later call. Each case runs in a child process, where the stand-in
is loaded before the library."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIP_INCLUDE = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "include"

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_largest.restype = C.c_size_t
refuse = lambda lo, hi: fake.fake_refuse(C.c_size_t(lo), C.c_size_t(hi))
launches = lambda part: fake.fake_launches(part.encode())
from voxgen_amd import abi, synth
from voxgen_amd.baselm import BaseLmEngine
from voxgen_amd.residual import ResidualFsqEngine
from voxgen_amd.runtime import Context, Model
ctx = Context(0)
def refused(call, *args):
    try:
        call(*args)
    except abi.VxError as e:
        return e.name
    return "VX_OK"
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not (HIP_INCLUDE / "hip" / "hip_runtime_api.h").exists():
        pytest.skip(f"no HIP headers under {HIP_INCLUDE}")
    out = tmp_path_factory.mktemp("fake") / "libfake_hip.so"
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-w", "-shared", "-fPIC", "-I", str(HIP_INCLUDE),
                    str(ROOT / "tests" / "fake_hip.c"), "-o", str(out)], check=True)
    return out


def child(fake, code):
    env = dict(os.environ, PYTHONPATH=str(ROOT))
    p = subprocess.run([sys.executable, "-c", PRELUDE + code, str(fake)], cwd=ROOT, env=env, text=True, timeout=120,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    assert p.returncode == 0, p.stdout[-3000:]


def test_refused_allocation_leaves_no_error_behind(fake):
    """The launch after a refused allocation is a launch like any other."""
    child(fake, """
refuse(1 << 20, 1 << 40)
assert refused(ctx.alloc, 1 << 20) == "VX_ERR_OOM"
refuse(0, 0)
b = ctx.alloc(4096)
b.fill_u32(7, 1024)
assert launches("k_fill_u32") == 1
""")


def test_prefill_without_room_for_the_f16_copy(fake):
    """The first batched prefill of an F16 engine whose prefill-layout copy is refused
    runs the general GEMM, and so does the next."""
    child(fake, """
cfg = synth.baselm_config(layers=2, hidden=256, ffn=512, vocab=64, q_heads=2, kv_heads=1, context_length=256,
                          active_context=256)
m = synth.build_baselm(cfg, seed=1, weight_type="f16")
model = Model(ctx, m.data, m.tensors)
copy = 2 * 2 * (2 * 256 * 256 + 2 * 128 * 256 + 3 * 512 * 256)   # the two layers' f16 matrices, less padding
eng = BaseLmEngine(ctx, model, cfg, strict_geometry=False)
refuse(copy, copy + 2 * 6 * 256)
for n in (37, 150):
    eng.prefill_tokens_batched_gpu_only([1] * n)
assert eng.position == 187
assert launches("k_repack_prefill") == 0 and launches("k_gemm_p") == 0 and launches("k_gemm") > 0
refuse(0, 0)
other = BaseLmEngine(ctx, model, cfg, strict_geometry=False)
other.prefill_tokens_batched_gpu_only([1] * 37)
assert launches("k_repack_prefill_f16") == 12 and launches("k_gemm_ps") == 8
""")


def test_text_prefix_workspace_refused_in_part(fake):
    """Each buffer of the ResidualLM's batched prefix refused in turn: the call fails,
    and the call after it, with room again, allocates what is missing and runs. The
    weight copy comes last, so that it cannot take the room of what is needed."""
    child(fake, """
cfg = synth.acoustic_config(layers=2, hidden=256, ffn=512, q_heads=2, kv_heads=1, latent=64, active_context=256)
m = synth.build_acoustic(cfg, seed=2)
model = Model(ctx, m.data, m.tensors)
rows = ctx.zeros(256 * 256 * 4)
copy = 2 * 2 * (2 * 256 * 256 + 2 * 128 * 256 + 3 * 512 * 256)
for part in ((256 * 512 * 4,) * 2, (256 * 256 * 4,) * 2, (4 << 20, 1 << 40)):   # fusion input, rows, workspace
    eng = ResidualFsqEngine(ctx, model, cfg, strict_geometry=False)
    repacks = launches("k_repack_prefill")
    refuse(*part)
    for _ in range(2):
        assert refused(eng.prefill_text_from_gpu_rows, rows, 37) == "VX_ERR_OOM"
    assert launches("k_repack_prefill") == repacks and eng.position == 0
    refuse(0, 0)
    eng.prefill_text_from_gpu_rows(rows, 37)
    assert launches("k_repack_prefill") == repacks + 12 and eng.position == 37
    eng.close()
eng = ResidualFsqEngine(ctx, model, cfg, strict_geometry=False)
before = launches("k_gemm_ps")
refuse(copy, copy + 2 * 6 * 256)
eng.prefill_text_from_gpu_rows(rows, 37)
assert eng.position == 37 and launches("k_gemm_ps") == before
""")


def test_baselm_prefill_token_buffer_refused(fake):
    """The BaseLM's token buffer refused after its workspace: the next call allocates it."""
    child(fake, """
cfg = synth.baselm_config(layers=1, hidden=256, ffn=512, vocab=64, q_heads=2, kv_heads=1, context_length=320,
                          active_context=320)
m = synth.build_baselm(cfg, seed=1, weight_type="f16")
model = Model(ctx, m.data, m.tensors)
eng = BaseLmEngine(ctx, model, cfg, strict_geometry=False)
refuse(320 * 4, 320 * 4)
assert refused(eng.prefill_tokens_batched_gpu_only, [1] * 5) == "VX_ERR_OOM"
refuse(0, 0)
eng.prefill_tokens_batched_gpu_only([1] * 5)
assert eng.position == 5
""")


def test_prefill_in_smaller_chunks_where_the_large_workspace_does_not_fit(fake):
    """Where the workspace of a whole chunk is refused, one of 512 rows is taken: 600
    positions are two chunks (two sets of layer launches), 600 with room are one."""
    child(fake, """
cfg = synth.baselm_config(layers=1, hidden=256, ffn=512, vocab=64, q_heads=2, kv_heads=1, context_length=4096,
                          active_context=4096)
m = synth.build_baselm(cfg, seed=1, weight_type="f16")
model = Model(ctx, m.data, m.tensors)
acfg = synth.acoustic_config(layers=1, hidden=256, ffn=512, q_heads=2, kv_heads=1, latent=64, active_context=4096)
am = synth.build_acoustic(acfg, seed=2)
amodel = Model(ctx, am.data, am.tensors)
rows = ctx.zeros(600 * 256 * 4)
def chunks(run):
    n = launches("k_prefill_attn")
    run()
    return launches("k_prefill_attn") - n
def base():
    eng = BaseLmEngine(ctx, model, cfg, strict_geometry=False)
    n = chunks(lambda: eng.prefill_tokens_batched_gpu_only([1] * 600))
    assert eng.position == 600
    return n
def residual():
    eng = ResidualFsqEngine(ctx, amodel, acfg, strict_geometry=False)
    n = chunks(lambda: eng.prefill_text_from_gpu_rows(rows, 600))
    assert eng.position == 600
    return n
fake.fake_largest()
assert base() == 1
whole = fake.fake_largest()   # the workspace
refuse(whole, 1 << 40)
assert base() == 2 and residual() == 2
refuse(2048 * 512 * 4, 2048 * 512 * 4)   # the fusion input of a whole chunk
assert residual() == 2
refuse(0, 0)
assert residual() == 1
""")


@pytest.mark.gpu
def test_refused_device_allocation_leaves_no_error_behind(ctx):
    """The same on the device: 2^50 bytes are more than any card has."""
    from voxgen_amd import abi
    with pytest.raises(abi.VxError) as e:
        ctx.alloc(1 << 50)
    assert e.value.name == "VX_ERR_OOM"
    b = ctx.alloc(4096)
    b.fill_u32(7, 1024)
    ctx.sync()
