"""What the C entries do on the host before, between and behind their launches, without a GPU: a child process loads tests/fake_hip.cpp in front of the library, so that every call of the HIP runtime
lands there -- which memory a copy would touch, on which device a thing is made, and errors where a test wants one."""
import os
import subprocess
import sys

import pytest

import wide_tiles
from powerserve_amd import hip

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes as C, sys
import numpy as np
fake = C.CDLL({fake!r}, mode=C.RTLD_GLOBAL)
fake.fake_stray.restype = fake.fake_held.restype = C.c_size_t
fake.fake_memory.argtypes = [C.c_size_t]
from powerserve_amd import hip, seqmodel, synth
def fail(name, n=1): fake.fake_fail(name.encode(), n)
def count(name): return fake.fake_count(name.encode())
def refused(f):
    try: f()
    except hip.PSHipError as e: return str(e)
    raise AssertionError("accepted")
L = synth.seq_layer
def quant(ctx, max_batch, preset="tiny-llama", n_ctx=1024):
    synth.write_model_dir({tmp!r} + "/quant", preset, 8, n_ctx=n_ctx, seed=1)
    return hip.Model(ctx, {tmp!r} + "/quant", max_batch=max_batch, n_ctx=n_ctx)
def seq(ctx, max_batch=8, vocab=30):
    cfg = synth.seq_config(24, vocab, [L("delta", 20, heads=4, kv_heads=2, dim=6, vdim=10, conv=4), L("wkv", None, heads=3, dim=8)], taps=3)
    synth.write_seq_model_dir({tmp!r} + "/seq", cfg, 1)
    return seqmodel.SeqModel(ctx, {tmp!r} + "/seq", max_batch=max_batch)
"""


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", so, os.path.join(HERE, "fake_hip.cpp")], check=True)
    return so


@pytest.fixture()
def child(fake, tmp_path):
    if not os.path.exists(hip.LIB_PATH):
        pytest.skip("lib/libps_hip.so not built")

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRELUDE.format(fake=fake, tmp=str(tmp_path)) + code + "\nprint('done', flush=True)\nimport os; os._exit(0)"], cwd=os.path.dirname(HERE),
                           capture_output=True, text=True, timeout=120)
        assert p.returncode == 0 and p.stdout.endswith("done\n"), (p.stdout[-1000:], p.stderr[-3000:])

    run.tmp = tmp_path
    return run


def test_more_wanted_rows_than_a_portion_holds_are_refused(child):
    """ps_hip_seq_forward: an index may repeat, but a portion's logits have max_batch rows; a longer list is refused before anything is launched."""
    child("""
ctx = hip.Ctx(0)
m = seq(ctx)
s = m.acquire()
fake.fake_reset()
for tokens, want in (([1], [0] * 9), ([1] * 20, [0, 1] + [9] * 9), ([1] * 20, [16] * 600)):
    refused(lambda: m.forward(s, tokens, want=want))
    assert count("hipLaunchKernel") == count("put_kernel") == count("hipMemcpyAsync") == 0 and m.position(s) == 0
m.forward(s, [1] * 20, want=[0] * 8 + [8] * 8 + [19] * 8)
assert m.position(s) == 20 and fake.fake_stray() == 0
""")


def test_ids_without_a_row_of_the_embedding_are_refused(child):
    """a table shorter than the vocabulary: an id that it has no row for is refused before anything is launched, one that it has is taken"""
    child("""
cfg = synth.seq_config(24, 30, [L("wkv", None, heads=3, dim=8)], taps=3)
t = synth.seq_tensors(cfg, 1)
t["embed"] = t["embed"][:20]
synth.write_seq_model_dir(".short", cfg, 1, t)
m = seqmodel.SeqModel(hip.Ctx(0), ".short", max_batch=8)
s = m.acquire()
fake.fake_reset()
for f in (lambda: m.forward(s, [19, 20]), lambda: m.forward(s, [29]), lambda: m.decode_greedy(s, 20, 3)):
    assert "outside the vocabulary" in refused(f)
assert count("hipLaunchKernel") == count("put_kernel") == 0
m.forward(s, [19, 0])
m.decode_greedy(s, 19, 3)
""".replace(".short", str(child.tmp / "short")))


def test_the_form_of_float32_matrices_does_not_depend_on_what_is_free(child):
    """ps_hip_dense_upload makes the form that it is asked for, and ps_hip_dense_f32_form chooses one by a model's size (tests/fake_hip.cpp: 1 GiB free of 288)"""
    child("""
ctx = hip.Ctx(0)
lib = ctx.L
bits = np.full((64, 64), 0x3f80, np.uint16)
def upload(form):
    h = C.c_void_p()
    ctx.check(lib.ps_hip_dense_upload(ctx.h, bits.ctypes.data_as(C.c_void_p), 64, 64, form, C.byref(h)))
    return h
for form, want in ((hip.DENSE_BF16, hip.DENSE_BF16), (hip.DENSE_F32, hip.DENSE_F32), (hip.DENSE_F32_LINES, hip.DENSE_F32_LINES), (7, hip.DENSE_F32), (-1, hip.DENSE_F32)):
    fake.fake_reset()
    h = upload(form)
    assert lib.ps_hip_dense_form(h) == want and count("hipMemGetInfo") == 0, form
    lib.ps_hip_dense_free(ctx.h, h)
for name in ("hipMemcpyAsync", "hipStreamSynchronize", "hipMalloc"):
    for nth in (1, 2):
        fake.fake_reset()
        fail(name, nth)
        if (name, nth) != ("hipStreamSynchronize", 2): refused(lambda: upload(hip.DENSE_F32_LINES))
for numbers, want in ((0, hip.DENSE_F32_LINES), (18 << 30, hip.DENSE_F32_LINES), ((18 << 30) + 1, hip.DENSE_F32), (1 << 50, hip.DENSE_F32)):
    assert lib.ps_hip_dense_f32_form(ctx.h, numbers) == want, numbers
fail("hipMemGetInfo")
assert lib.ps_hip_dense_f32_form(ctx.h, 1) == hip.DENSE_F32
cfg = synth.seq_config(64, 30, [L("wkv", None, heads=1, dim=64)], taps=3)
synth.write_seq_model_dir(".dir", cfg, 1)
for dtype, form, want in (("bfloat16", None, hip.DENSE_BF16), ("float32", None, hip.DENSE_F32_LINES), ("float32", hip.DENSE_F32, hip.DENSE_F32), ("bfloat16", hip.DENSE_F32, hip.DENSE_BF16)):
    m = seqmodel.SeqModel(ctx, ".dir", dtype=dtype, max_batch=8, f32_form=form)
    assert {lib.ps_hip_dense_form(w) for w in m._up.mats} == {want}, (dtype, form)
    m.close()
""".replace(".dir", str(child.tmp / "dir")))


def test_a_joint_projection_without_room_for_its_second_form(child):
    """ps_hip_seq_create: of all the memory a float32 model asks for, the bfloat16 form of two mixers' joint projection is the one piece that it can do without; a portion's products then run as fp32 ones"""
    child("""
ctx = hip.Ctx(0)
att = {"heads": 8, "kv_heads": 1, "dim": 64, "vdim": 64, "mask": {"size": 9, "pool": 3}, "rot": {"base": 100.0, "dims": 8}, "scale": 0.2}
cfg = synth.parallel_config(1024, 30, [synth.parallel_layer(None, att, {"heads": 8, "dim": 64, "vdim": 64, "tau": 4.0}, 1.0, 0.5)], taps=2)
synth.write_seq_model_dir(".dir", cfg, 1)
def load(): return seqmodel.SeqModel(ctx, ".dir", dtype="float32", max_batch=200, launch_rows=200)
fake.fake_reset()
load().close()
took = []
for n in range(1, count("hipMalloc") + 1):
    fake.fake_reset()
    fail("hipMalloc", n)
    try: m = load()
    except hip.PSHipError: continue
    s = m.acquire()
    fake.fake_reset()
    m.forward(s, [1] * 200, want=[199])
    took.append((count("dense_mm_ring_kernelIf"), count("dense_mm_ring_kernelIt"), fake.fake_stray()))
    m.close()
fake.fake_reset()
m = load()
s = m.acquire()
fake.fake_reset()
m.forward(s, [1] * 200, want=[199])
f32, lines = count("dense_mm_ring_kernelIf"), count("dense_mm_ring_kernelIt")
assert lines > 0 and took == [(f32 + 1, lines - 1, 0)], (took, f32, lines)
""".replace(".dir", str(child.tmp / "dir")))


def test_a_model_without_room_for_wide_launch_sequences(child):
    """ps_hip_seq_create: launch sequences of four times max_batch where the memory is there, of max_batch where it is not; more wanted rows than the head takes at a time go in groups"""
    child("""
ctx = hip.Ctx(0)
toks, want = [1] * 300, list(range(300))
fake.fake_reset()
m = seq(ctx, 64)
allocations = count("hipMalloc")
s = m.acquire()
fake.fake_reset()
m.forward(s, toks, want=want)
assert count("seq_set_step_kernel") == 2 and count("dense_argmax_kernel") == 5 and m.position(s) == 300 and fake.fake_stray() == 0
for n in (0, 1, 7): # (the last ones are the model's own)
    fail("hipMalloc", allocations - n)
    m = seq(ctx, 64)
    s = m.acquire()
    fake.fake_reset()
    m.forward(s, toks, want=want)
    assert count("seq_set_step_kernel") == 5 and count("dense_argmax_kernel") == 5 and m.position(s) == 300 and fake.fake_stray() == 0
""")


def test_what_wide_launch_sequences_may_take(child):
    """ps_hip_seq_create: four times max_batch tokens where that takes at most a 64th of the device's memory beyond what max_batch does, else twice as many, else max_batch; the rings of all slots are
    part of it.  ps_hip_seq_create_sized makes the size that it is asked for"""
    child("""
ctx = hip.Ctx(0)
cfg = synth.seq_config(24, 30, [L("latent_attention", 20, heads=2, dim=8, vdim=8, q_rank=8, kv_rank=16, rot={"base": 1e4, "dims": 8}, rot_dim=8, mask={"size": 9}, scale=0.3), L("wkv", None, heads=3, dim=8)], taps=3)
synth.write_seq_model_dir(".dir", cfg, 1)
def load(slots=2, rows=0, batch=64, context=0):
    m = seqmodel.SeqModel(ctx, ".dir", max_batch=batch, n_slots=slots, launch_rows=rows, max_context=context)
    held, r, slot = fake.fake_held(), m.launch_rows, m.slot_bytes
    s = m.acquire()
    fake.fake_reset()
    m.forward(s, [1] * 300, want=[0, 299])
    assert count("seq_set_step_kernel") == -(-300 // r) and fake.fake_stray() == 0
    m.close()
    return r, held, slot
bytes_ = {(n, r): load(n, r) for n in (2, 40) for r in (64, 128, 256)}
for (n, r), (rows, held, slot) in bytes_.items(): assert rows == r and slot - bytes_[n, 64][2] == (r - 64) * (16 + 8) * 4
for n in (2, 40):
    extra = {r: bytes_[n, r][1] - bytes_[n, 64][1] for r in (128, 256)}
    for spare, want in ((extra[256], 256), (extra[256] - 1, 128), (extra[128], 128), (extra[128] - 1, 64), (0, 64)):
        fake.fake_memory(64 * spare)
        assert load(n)[0] == want, (n, spare)
        for r in (64, 128, 256, 200): assert load(n, r)[0] == r
fake.fake_memory(288 << 30)
fake.fake_reset()
fail("hipMemGetInfo")
assert load()[0] == 64
for batch, context, want in ((63, 0, 63), (64, 400, 256), (128, 400, 400), (600, 0, 2048), (3000, 0, 3000)): assert load(batch=batch, context=context)[0] == want, batch
assert "launch_rows" in refused(lambda: load(rows=63))
""".replace(".dir", str(child.tmp / "dir")))


def test_images_of_the_split_attention_have_a_bound(child):
    """a window of everything behind many heads: their images may take a 64th of the device's memory, beyond that the fp32 form attends"""
    child("""
ctx = hip.Ctx(0)
cfg = synth.seq_config(64, 30, [L("latent_attention", None, heads=80, dim=128, vdim=128, q_rank=8, kv_rank=16, rot={"base": 1e4, "dims": 8}, rot_dim=64, mask={"size": 3000}, scale=0.3)], taps=1)
synth.write_seq_model_dir(".dir", cfg, 1)
def load():
    m = seqmodel.SeqModel(ctx, ".dir", max_batch=128, n_slots=1, launch_rows=128, max_context=3000)
    held, s = fake.fake_held(), m.acquire()
    fake.fake_reset()
    m.forward(s, [1] * 128)
    took = count("split_attn_kernel"), count("latent_attn_mfma_kernel")
    m.close()
    return held, took
with_, took = load()
fake.fake_memory(0)
without, plain = load()
assert took == (1, 0) and plain == (0, 1) and with_ > without
for spare, want in ((with_ - without, took), (with_ - without - 1 - 256, plain)):
    fake.fake_memory(64 * spare)
    assert load()[1] == want
""".replace(".dir", str(child.tmp / "dir")))


def test_portions_whose_attention_is_split(child):
    """k_splitattn.hip takes 80 work-groups of 128 rows and more, and more than 512 of 16: 129 rows of 64 heads and 193 of 40, not 128, 192 or 256 of 39, nor a single row of many heads; keys of 128
    and 192 numbers, values of 128"""
    child("""
ctx = hip.Ctx(0)
def took(tokens, heads, dim=128, vdim=128):
    cfg = synth.zusolix_config(64, 30, [synth.zusolix_layer("attention", synth.zusolix_attention(heads, 1, dim, vdim, 0.1))])
    synth.write_seq_model_dir(".dir", cfg, 1)
    m = seqmodel.SeqModel(ctx, ".dir", max_batch=300, n_slots=1, max_context=400)
    s = m.acquire()
    fake.fake_reset()
    m.forward(s, [1] * tokens)
    n = count("split_keys_kernel"), count("split_attn_kernel"), count("winattn_mfma_kernel")
    m.close()
    return n
for sizes in ((129, 64), (193, 40), (97, 80), (65, 128), (257, 32), (129, 64, 192)): assert took(*sizes) == (1, 1, 0), sizes
for sizes in ((128, 64), (192, 40), (96, 80), (64, 128), (256, 39), (256, 32), (1, 80), (2, 128), (1, 200), (129, 64, 160), (129, 64, 128, 96)): assert took(*sizes)[:2] == (0, 0), sizes
""".replace(".dir", str(child.tmp / "dir")))


def test_portions_whose_rows_several_work_groups_share(child):
    """k_splitattn.hip sa_plan_of: where whole tiles of 128 rows leave CUs waiting -- fewer tiles than CUs behind many keys -- their parts are joined; tiles of a few blocks and many tiles stay whole"""
    child("""
ctx = hip.Ctx(0)
def joined(tokens, heads, behind=0):
    cfg = synth.zusolix_config(64, 30, [synth.zusolix_layer("attention", synth.zusolix_attention(heads, 1, 128, 128, 0.1))])
    synth.write_seq_model_dir(".dir", cfg, 1)
    m = seqmodel.SeqModel(ctx, ".dir", max_batch=1500, n_slots=1, max_context=3000)
    s = m.acquire()
    if behind: m.forward(s, [1] * behind)
    fake.fake_reset()
    m.forward(s, [1] * tokens)
    assert count("split_attn_kernel") == 1
    n = count("split_join_kernel")
    m.close()
    return n
for sizes in ((1400, 16), (129, 64, 1000), (700, 32)): assert joined(*sizes) == 1, sizes
for sizes in ((129, 64), (400, 64), (1024, 128)): assert joined(*sizes) == 0, sizes
""".replace(".dir", str(child.tmp / "dir")))


@pytest.mark.parametrize("dtype,rank,folds", [("bfloat16", 1, 1), ("bfloat16", 24, 1), ("bfloat16", 25, 0), ("bfloat16", 32, 1), ("bfloat16", 40, 0), ("bfloat16", 64, 0), ("float32", 24, 1), ("float32", 25, 0), ("float32", 32, 0)])
def test_a_tokens_decay_inside_its_scan(child, dtype, rank, folds):
    """seqmodel.hip: the decay's second product and the copy of the token's input are launches of their own for the ranks where those are the faster ones"""
    child("""
ctx = hip.Ctx(0)
cfg = synth.seq_config(64, 30, [L("wkv", None, heads=2, dim=32)], taps=2)
synth.write_seq_model_dir(".dir", cfg, 1, synth.seq_tensors(cfg, 1, RANK))
m = seqmodel.SeqModel(ctx, ".dir", dtype="DTYPE", max_batch=8)
s = m.acquire()
fake.fake_reset()
m.forward(s, [1])
assert (count("sq_decay_scan_kernelILi0ELi1ELb1E"), count("sq_decay_scan_kernelILi0ELi1ELb0E")) == (FOLDS, 1 - FOLDS)
""".replace(".dir", str(child.tmp / "dir")).replace("RANK", str(rank)).replace("DTYPE", dtype).replace("FOLDS", str(folds)))


@pytest.mark.parametrize("heads,norms,itself", [(8, "heads", 1), (24, "heads", 1), (26, "heads", 0), (36, "none", 1), (36, "whole", 0)])
def test_a_token_whose_attention_makes_its_own_row(child, heads, norms, itself):
    """seqmodel.hip: without norms, or with those of every head and up to twelve heads a group; more, and norms over whole projections, have the preparation's launch in front"""
    child("""
ctx = hip.Ctx(0)
if NORMS == "heads":
    cfg = synth.pupidra_config(64, 30, [synth.pupidra_layer("attention", synth.pupidra_attention(HEADS, 2, 32, 32, 1.0, 9, 20))])
else:
    at = {"heads": HEADS, "kv_heads": 2, "dim": 32, "vdim": 32, "mask": {"size": 5, "pool": 3}, "rot": {"base": 100.0, "dims": 16}, "scale": 0.2}
    cfg = synth.parallel_config(64, 30, [synth.parallel_layer(None, at, {"heads": 1, "dim": 16, "vdim": 16, "tau": 4.0}, 1.0, 0.5)], taps=2)
t = {n: v for n, v in synth.seq_tensors(cfg).items() if NORMS != "none" or not n.endswith(("q.norm", "k.norm"))}
synth.write_seq_model_dir(".dir", cfg, 1, t)
m = seqmodel.SeqModel(ctx, ".dir", max_batch=8, n_slots=1, max_context=100)
s = m.acquire()
fake.fake_reset()
m.forward(s, [1])
assert (count("winattn_step_kernel"), count("winattn_prep_kernel")) == (1, 1 - ITSELF)
""".replace(".dir", str(child.tmp / "dir")).replace("HEADS", str(heads)).replace("NORMS", repr(norms)).replace("ITSELF", str(itself)))


def test_tiles_of_several_parts_are_joined(child):
    """k_splitattn.hip sa_plan_of: the portions whose results tests/test_gpu_seq.py compares -- 41 heads in parts in both portions, 81 in whole tiles"""
    child("""
ctx = hip.Ctx(0)
def joined(cfg):
    synth.write_seq_model_dir(".dir", cfg, 1)
    m = seqmodel.SeqModel(ctx, ".dir", dtype="float32", max_batch=260, n_slots=1, max_context=500)
    s, n = m.acquire(), []
    for T in (260, 200):
        fake.fake_reset()
        m.forward(s, [1] * T)
        n.append((count("split_attn_kernel"), count("split_join_kernel")))
    m.close()
    return n
latent = lambda heads: synth.pupidra_config(64, 30, [synth.pupidra_layer("latent_attention", synth.pupidra_latent(heads, 96, 32, 128, 32, 0.1, 1e4))])
assert joined(latent(41)) == [(1, 1), (1, 1)]
assert joined(latent(81)) == [(1, 0), (1, 0)]
assert joined(synth.zusolix_config(64, 30, [synth.zusolix_layer("attention", synth.zusolix_attention(41, 1, 128, 128, 0.1, 5.0, (0.4, 7)), ff=64)])) == [(1, 1), (1, 1)]
""".replace(".dir", str(child.tmp / "dir")))


def test_the_tiles_of_wide_products(child):
    """k_dense.hip dn_ring_plan: the tile and the parts of every product of wide_tiles.py, by the launch's name"""
    products = [(fmt, T, N, K, wide_tiles.kernel(fmt, BM, BN, int(N % 4 != 0)), f"dense_mm_sum_kernelILi{BM}ELi{BN}E", S) for (fmt, BM, BN), sizes in wide_tiles.PRODUCTS.items() for T, N, K, S in sizes]
    child("""
ctx = hip.Ctx(0)
bits = np.zeros(26 << 20, np.uint16)
wrong = []
for fmt, T, N, K, kernel, sums, S in PRODUCTS:
    w = C.c_void_p()
    form = hip.DENSE_BF16 if fmt == "bfloat16" else hip.DENSE_F32_LINES
    x, o = hip.DevArray(ctx, (T, K), np.float32), hip.DevArray(ctx, (T, N), np.float32)
    ctx.check(ctx.L.ps_hip_dense_upload(ctx.h, bits.ctypes.data_as(C.c_void_p), N, K, form, C.byref(w)))
    fake.fake_reset()
    ctx.check(ctx.L.ps_hip_dense_matmul(ctx.h, w, x.ptr, T, o.ptr, 1.0))
    if (count(kernel), count(sums)) != (1, int(S > 1)): wrong.append((fmt, T, N, K, kernel, count(kernel), count(sums)))
    ctx.L.ps_hip_dense_free(ctx.h, w)
    x.free(); o.free()
assert not wrong, "\\n".join(map(str, wrong))
""".replace("PRODUCTS", repr(products)))


def test_the_tiles_of_products_with_an_epilogue(child):
    """the same of the models of wide_tiles.EPILOGUES: one launch of the named kernel in their portion"""
    models = [(which, fmt, size, T, width, wide_tiles.kernel(fmt, BM, BN, 0), f"dense_mm_sum_kernelILi{BM}ELi{BN}E", S) for (which, fmt), cases in wide_tiles.EPILOGUES.items() for size, T, width, BM, BN, S in cases]
    child("""
sys.path.insert(0, TESTS)
import wide_tiles
ctx = hip.Ctx(0)
wrong = []
for which, fmt, size, T, width, kernel, sums, S in MODELS:
    synth.write_seq_model_dir(".dir", wide_tiles.layers(synth, which, size, width), 1)
    m = seqmodel.SeqModel(ctx, ".dir", dtype=fmt, max_batch=T, n_slots=1, max_context=T + 100, f32_form=hip.DENSE_F32_LINES if fmt == "float32" else None)
    s = m.acquire()
    fake.fake_reset()
    m.forward(s, [1] * T)
    if (count(kernel), count(sums)) != (1, S): wrong.append((which, fmt, size, T, width, kernel, count(kernel), count(sums)))
    m.close()
assert not wrong, "\\n".join(map(str, wrong))
""".replace("TESTS", repr(HERE)).replace("MODELS", repr(models)).replace(".dir", str(child.tmp / "dir")))


@pytest.mark.parametrize("width,experts,ff,tokens", [(1024, 64, 768, 9), (2048, 8, 1536, 150)])
def test_the_tiles_of_experts(child, width, experts, ff, tokens):
    """k_dense.hip dn_mean_row_tiles: 18 slots of 64 matrices are 16 tiles of 64 rows, 300 slots of eight are eight -- one round of 64 x 64 tiles, not the start of a second one"""
    child("""
ctx = hip.Ctx(0)
cfg = synth.pupidra_config(WIDTH, 30, [synth.pupidra_layer("attention", synth.pupidra_attention(2, 1, 16, 16, 0.3, 9, 2), moe=(EXPERTS, 2, FF, 1.7), shared=8)])
synth.write_seq_model_dir(".dir", cfg, 1)
m = seqmodel.SeqModel(ctx, ".dir", max_batch=TOKENS, n_slots=1, max_context=400)
s = m.acquire()
fake.fake_reset()
m.forward(s, [1] * TOKENS)
assert count("dense_mm_ring_kernelItLi64ELi64E") >= 2 and count("dense_mm_ring_kernelItLi64ELi128E") == 0
""".replace(".dir", str(child.tmp / "dir")).replace("WIDTH", str(width)).replace("EXPERTS", str(experts)).replace("FF", str(ff)).replace("TOKENS", str(tokens)))


def test_the_measured_products_of_experts_are_the_ones_that_run(child):
    """ps_hip_seq_bench_kernel: a portion's second product of the experts reads the rounded rows of the first one, in a step and where it is measured"""
    child("""
ctx = hip.Ctx(0)
for ff in (128, 72): # (72: no whole blocks, the tiled kernel)
    cfg = synth.pupidra_config(64, 30, [synth.pupidra_layer("attention", synth.pupidra_attention(2, 1, 16, 16, 0.3, 9, 2), moe=(5, 2, ff, 1.7), shared=None)])
    synth.write_seq_model_dir(".dir", cfg, 1)
    m = seqmodel.SeqModel(ctx, ".dir", max_batch=64)
    us, by, fl = C.c_double(), C.c_double(), C.c_double()
    def packed(which, reps):
        fake.fake_reset()
        ctx.check(ctx.L.ps_hip_seq_bench_kernel(m.h, which, 64, reps, C.byref(us), C.byref(by), C.byref(fl)))
        return count("dense_pack_kernel")
    for which, want in ((2, 1), (3, 0)): assert packed(which, 5) - packed(which, 2) == 3 * want, (ff, which)
""".replace(".dir", str(child.tmp / "dir")))


def test_copies_to_the_host_keep_their_error_cases(child):
    """ps_hip_memcpy_d2h: what a kernel could not read without a fault is left to the runtime's copy, whatever that says"""
    child("""
ctx, other = hip.Ctx(0), hip.Ctx(1)
out = np.zeros(256, np.float32)
def d2h(dst, src, n): ctx.check(ctx.L.ps_hip_memcpy_d2h(ctx.h, dst, src, n))
p, q, far = ctx.malloc(1024), ctx.malloc(1024), other.malloc(1024)
fake.hipSetDevice(0)
fake.fake_reset()
for dst, src, n in ((out.ctypes.data, None, 64), (out.ctypes.data, p, 1028), (out.ctypes.data, p + 512, 1024), (None, p, 64), (out.ctypes.data, 4096, 64)):
    refused(lambda: d2h(dst, src, n))
d2h(out.ctypes.data, far, 1024)
d2h(q, p, 1024)
assert count("pin_copy_kernel") == 0 and count("hipMemcpyAsync") == 7 and fake.fake_stray() == 0
d2h(out.ctypes.data, p + 512, 512)
assert count("pin_copy_kernel") == 1 and count("hipMemcpyAsync") == 7 and fake.fake_stray() == 0
d2h(out.ctypes.data, p + 2, 64)
d2h(out.ctypes.data, p, 1023)
d2h(out.ctypes.data, p, 0)
""")


def test_results_through_pinned_memory_by_size(child):
    """a copy that is waited for up to 20 KB, where the runtime's is the slower one; a portion's rows, which come behind its launches, up to a half of the pinned memory"""
    child("""
ctx = hip.Ctx(0)
p, out = ctx.malloc(1 << 20), np.zeros(1 << 18, np.float32)
for n, kernel in ((4, 1), (20480, 1), (20484, 0), (65536, 0), (1 << 20, 0)):
    fake.fake_reset()
    ctx.check(ctx.L.ps_hip_memcpy_d2h(ctx.h, out.ctypes.data, p, n))
    assert (count("pin_copy_kernel"), count("hipMemcpyAsync")) == (kernel, 1 - kernel), n
m = seq(ctx, 8, 100000)
s = m.acquire()
for tokens, want, kernels, copies in ((8, 5, 1, 0), (8, 6, 0, 1), (16, 13, 1, 1)):
    fake.fake_reset()
    m.forward(s, [1] * tokens, want=np.arange(want))
    assert (count("pin_copy_kernel"), count("hipMemcpyAsync")) == (kernels, copies), (tokens, want)
""")


def test_pinned_memory_and_its_events_are_made_on_the_contexts_device(child):
    """two contexts: copies on the first while the second's device is current (before and after there is pinned memory), then portions on the first, whose events have to be the first's"""
    child("""
ctx = hip.Ctx(0)
m = seq(ctx, 8, 3000)
s, p, out = m.acquire(), ctx.malloc(64), np.zeros(16, np.float32)
other = hip.Ctx(1)
fake.fake_reset()
for _ in range(2):
    fake.hipSetDevice(1)
    ctx.check(ctx.L.ps_hip_memcpy_d2h(ctx.h, out.ctypes.data, p, 64))
    m.forward(s, [1] * 16, want=np.arange(16))
assert count("hipEventRecord") == 4 and count("hipMemcpyAsync") == 2
""")


def test_a_slots_position_follows_its_state_when_a_later_portion_fails(child):
    """the recurrent states move with every portion that was launched, whatever becomes of its results: so does the position, and nothing is still on its way to the caller's memory"""
    child("""
ctx = hip.Ctx(0)
m = seq(ctx, 8, 3000)
for name, nth in (("hipEventSynchronize", 1), ("hipEventSynchronize", 2), ("hipEventRecord", 1), ("hipEventRecord", 3), ("hipStreamSynchronize", 1)):
    s = m.acquire()
    fake.fake_reset()
    fail(name, nth)
    refused(lambda: m.forward(s, [1] * 32, want=np.arange(32)))
    ran = count("seq_set_step_kernel")
    assert ran and m.position(s) == 8 * ran and count("hipStreamSynchronize"), (name, nth, ran, m.position(s))
    at = m.position(s)
    m.forward(s, [1] * 9, want=[8])
    assert m.position(s) == at + 9
    m.release(s)
s = m.acquire()
fake.fake_reset()
fail("hipGetLastError", 2)
refused(lambda: m.forward(s, [1] * 32))
assert m.position(s) == 8 * (count("seq_set_step_kernel") - 1) == 8  # (a portion whose launches failed has not been taken)
""")


def test_inputs_travel_as_arguments_up_to_a_size_and_their_errors_come_back(child):
    """csrc/ctx.hip ps_put: a large tree's mask is one copy, not 75 launches; a launch that fails ends the call"""
    child("""
ctx = hip.Ctx(0)
m = quant(ctx, 512)
for n, launches in ((12, 1), (139, 6), (140, 0), (512, 0)):
    t = np.arange(n) % 500
    see = np.tril(np.ones((n, n), np.uint8))
    fake.fake_reset()
    m.forward_tree(t, np.arange(n), see)
    assert (count("put_kernel"), count("hipMemcpyAsync")) == (launches, 0 if launches else 3), (n, count("put_kernel"), count("hipMemcpyAsync"))
    assert fake.fake_stray() == 0
q = seq(ctx)
s = q.acquire()
for f in (lambda: m.forward_tree([1, 2], [0, 1], np.tril(np.ones((2, 2), np.uint8))), lambda: m.forward_tree(np.arange(500), np.arange(500), np.ones((500, 500), np.uint8)),
          lambda: m.forward([1, 2], [0, 1]), lambda: m.prefill(np.arange(20), 10), lambda: m.decode_greedy(1, 3), lambda: q.forward(s, [1, 2])):
    fake.fake_reset()
    f()
    m.kv_rollback(m.position)
    at = q.position(s)
    for name in ("put_kernel", "hipMemcpyAsync"):
        fake.fake_reset()
        fail(name)
        try: f()
        except hip.PSHipError: assert m.position == 0 and q.position(s) == at
        else: assert name == "hipMemcpyAsync" or not count(name), name
        m.kv_rollback(m.position)
        at = q.position(s)
""")


@pytest.mark.parametrize("arch,heads,kv,size,line", [("qwen2", 16, 4, 64, 880), ("qwen2", 14, 2, 64, 3300), ("qwen2", 8, 8, 128, 220), ("qwen2", 40, 8, 128, 1350), ("llama", 24, 8, 96, 390),
                                                     ("llama", 32, 32, 128, 1160), ("llama", 40, 8, 128, 250), ("llama", 16, 4, 64, 0)])
def test_single_token_attention_by_the_length_a_call_comes_to(child, arch, heads, kv, size, line):
    """attn_decode1_kernel up to a cache length (k_attn.hip psl_attn_decode1_until): eager and captured single tokens and greedy calls on both sides of it.  A captured step that holds the kernel is
    dropped by the first call that would outgrow the line, a step without it stays; every layer of every token takes the one or the other."""
    child("""
arch, heads, kv, size, line = %r
synth.PRESETS["one"] = (arch, heads * size, 256, 2, heads, kv, size, 512, 1e4, 2 if arch == "qwen2" else 0, True, 1e-5)
ctx = hip.Ctx(0)
m = quant(ctx, 64, "one", 3600)
def took(f, at):
    if m.position > at: m.kv_rollback(m.position - at)
    if m.position < at: m.prefill(np.ones(at - m.position, int), 64)
    fake.fake_reset()
    f()
    n, all_ = count("attn_decode1_kernel"), count("attn_decode1_kernel") + count("attn_decode2_kernel") + count("attn_softmax_pv_kernel")
    return n, all_, count("hipStreamBeginCapture")
def same(got, want): assert got[:len(want)] == want, (mode, got, want)
greedy = lambda n: lambda: m.decode_greedy(1, n)
token = lambda: m.forward([1], [m.position])
for mode in (0, 1):
    m.set_mode(mode)
    if line:
        at = line - 40
        same(took(greedy(8), at), (16, 16))
        same(took(greedy(32), at + 8), (64, 64, 0))     # to the line: replayed
        same(took(greedy(33), at + 8), (0, 66, 1 - mode))
        same(took(greedy(4), at + 8), (8 * mode, 8, 0))    # (a step without it is kept)
        same(took(token, line - 1), (2, 2))
        same(took(token, line - 1), (2, 2, 0))
    at = max(line, 8)
    same(took(token, at), (0, 2))
    same(took(token, at), (0, 2, 0))
    same(took(greedy(4), at), (0, 8))
    m.kv_rollback(m.position)
""" % ((arch, heads, kv, size, line),))



def test_a_captured_step_is_made_again_when_its_hint_is_far_behind(child):
    """csrc/model.hip plan_outlived: a plan with attn_decode1_kernel made behind 100 positions outlives 246 by 31 tokens, greedy or one by one; one made behind 480, and one without the kernel, by 1024"""
    child("""
def go(preset, lines):
    m = quant(ctx, 64, preset, 3600)
    def made(f, at):
        if m.position > at: m.kv_rollback(m.position - at)
        if m.position < at: m.prefill(np.ones(at - m.position, int), 64)
        fake.fake_reset()
        f()
        return count("hipStreamBeginCapture")
    greedy = lambda n: lambda: m.decode_greedy(1, n)
    token = lambda: m.forward([1], [m.position])
    for at, n, want in lines: assert made(greedy(n), at) == want, (preset, at, n)
    m.kv_rollback(m.position)
    for at, n, want in lines: assert sum(made(token, at) for _ in range(n)) == want, (preset, at, n)
    m.close()
synth.PRESETS["with"] = ("qwen2", 14 * 64, 256, 1, 14, 2, 64, 512, 1e4, 2, True, 1e-5)
synth.PRESETS["without"] = ("llama", 16 * 64, 256, 1, 16, 4, 64, 512, 1e4, 0, True, 1e-5)
ctx = hip.Ctx(0)
go("with", [(100, 1, 1), (200, 40, 0), (245, 1, 0), (246, 16, 0), (300, 15, 0), (300, 1, 1), (300, 40, 0), (545, 40, 0), (546, 40, 1), (1569, 40, 0), (1570, 1, 1), (0, 1, 1), (95, 1, 0), (96, 32, 1)])
go("without", [(100, 1, 1), (300, 40, 0), (1123, 1, 0), (1124, 1, 1), (480, 1, 1), (1503, 1, 0), (1504, 1, 1)])
""")


WIDE = {"wide-8": (64, 8, 32, 8), "wide-16": (32, 32, 96, 16), "wide-32-of-96": (48, 48, 96, 32), "wide-32-of-32": (136, 17, 32, 32), "wide-64": (136, 17, 64, 64)}  # heads, kv heads, size, channels


@pytest.mark.parametrize("heads,kv,size,channels", WIDE.values(), ids=WIDE.keys())
def test_channels_per_work_group_of_the_single_token_attention(child, heads, kv, size, channels):
    """four channels of a head per work-group where all of them then fit on 256 CUs, else as many more as it takes: the shapes that tests/test_gpu_model.py runs have the widths it says"""
    child("""
heads, kv, size, channels = %r
synth.PRESETS["one"] = ("llama", heads * size, 128, 1, heads, kv, size, 128, 1e4, 0, True, 1e-5)
ctx = hip.Ctx(0)
m = quant(ctx, 8, "one", 64)
m.forward([1], [0])
assert fake.fake_blocks(b"attn_decode1_kernel") == heads * size // channels
""" % ((heads, kv, size, channels),))
