"""Layer-list models on the GPU against the plain float64 statement in tests/seq_oracle.py: small configurations and random weights made
here, every schedule (whole prompts, token by token, portions, interleaved requests, reused slots, ring wrap, greedy generation)."""
import numpy as np
import pytest

import seq_oracle
import wide_tiles
from powerserve_amd import hip, host, seqmodel, synth
from powerserve_amd.safetensors_io import f32_to_bf16_bits

pytestmark = pytest.mark.gpu

L = synth.seq_layer
LAT = dict(rot={"base": 10000.0, "dims": 8}, rot_dim=8)
CONFIGS = {
    # sizes that are multiples of nothing in particular; unequal taps; a layer without feed-forward
    "mixed": synth.seq_config(48, 64, [L("wkv", 40, heads=2, dim=24), L("delta", None, heads=4, kv_heads=2, dim=12, vdim=20, conv=4),
                                       L("latent_attention", 56, heads=3, dim=16, vdim=24, q_rank=20, kv_rank=28, mask={"size": 9}, scale=0.3, **LAT)],
                              taps=2, logit_scale=0.5),
    # sizes on the matrix cores' grid, other order of layers
    "aligned": synth.seq_config(128, 96, [L("latent_attention", 192, heads=2, dim=32, vdim=64, q_rank=48, kv_rank=64, mask={"size": 33}, scale=0.125,
                                            rot={"base": 500.0, "dims": 16}, rot_dim=16),
                                          L("delta", 128, heads=2, kv_heads=2, dim=64, vdim=32, conv=3), L("wkv", 128, heads=2, dim=64)], taps=3, eps=1e-5),
    # heads of more than 64 rows (state rows spread over 8 and 16 lanes), one head, one tap (no tail at all), window of one
    "wide_heads": synth.seq_config(80, 50, [L("wkv", 32, heads=1, dim=80), L("delta", 32, heads=3, kv_heads=1, dim=144, vdim=72, conv=1),
                                            L("latent_attention", None, heads=1, dim=8, vdim=70, q_rank=9, kv_rank=11, mask={"size": 1}, scale=1.0,
                                              rot={"base": 100.0, "dims": 2}, rot_dim=6)], taps=1),
    "wkv": synth.seq_config(40, 32, [L("wkv", None, heads=2, dim=20)], taps=4),
    "delta": synth.seq_config(40, 32, [L("delta", None, heads=2, kv_heads=1, dim=20, vdim=12, conv=2)], taps=3),
    "latent": synth.seq_config(40, 32, [L("latent_attention", None, heads=2, dim=12, vdim=20, q_rank=16, kv_rank=24, mask={"size": 6}, scale=0.4, **LAT)], taps=3),
    "ff": synth.seq_config(40, 32, [L("wkv", 24, heads=1, dim=8)], taps=2),
}
# float32: a few ulps of fp32 sums.  bfloat16: the operands of every matrix product are rounded to 8 bits of mantissa, which in models this
# narrow (48 to 128 channels) leaves 1-3 % on a typical row and up to 7 % on the worst of a hundred rows, whatever the schedule
TOL = {"float32": 2e-4, "bfloat16": 1e-1}
# what ps_hip_dense_upload makes of a matrix: fp32 on the fp32 instruction, fp32 on the bf16 instruction (three lines of the operand), bf16
FORMS = {"float32": hip.DENSE_F32, "float32 lines": hip.DENSE_F32_LINES, "bfloat16": hip.DENSE_BF16}


def err(got, want):
    """centred rms of the difference over the rms of the logits, worst row"""
    d = np.asarray(got, dtype=np.float64) - want
    d = d - d.mean(-1, keepdims=True)
    s = np.sqrt(np.mean((want - want.mean(-1, keepdims=True)) ** 2))
    return float(np.sqrt(np.mean(d * d, -1)).max() / s)


@pytest.fixture(scope="module")
def made(ctx, tmp_path_factory):
    """(name, dtype, max_batch) -> (model, cfg, tensors); models are built once and closed at the end"""
    cache = {}

    def get(name, dtype="float32", max_batch=16, seed=0, cfg=None, tensors=None):
        key = (name, dtype, max_batch, seed)
        if key not in cache:
            c = cfg or CONFIGS[name]
            d = str(tmp_path_factory.mktemp("m"))
            t = synth.write_seq_model_dir(d, c, seed, tensors)
            cache[key] = (seqmodel.load_model(ctx, d, dtype=dtype, max_batch=max_batch, n_slots=3), c, t)
        return cache[key]

    yield get
    for m, _, _ in cache.values():
        m.close()


def tokens_for(cfg, n, seed=1):
    return np.random.default_rng(seed).integers(0, cfg["vocab"], n).astype(np.int32)


def run_portions(m, toks, sizes):
    """the sequence cut into portions of the given sizes (cycled), all logits"""
    s, out, at, i = m.acquire(), [], 0, 0
    while at < len(toks):
        n = min(sizes[i % len(sizes)], len(toks) - at)
        out.append(m.forward(s, toks[at:at + n], np.arange(n)))
        at, i = at + n, i + 1
    m.release(s)
    return np.concatenate(out)


# a portion's boundaries in one launch each (k_seqmix.hip sq_boundary_rows_kernel): portions of fewer tokens than the filter reaches back, whole and begun work-groups of three rows and of four (from 513
# on), single tokens in between (a launch of their own, over the same tail), long rows of few tokens (as before: a launch each); rows that end inside a wave, in one of sixteen waves; a layer without feed-forward; the layers' results as well
@pytest.mark.parametrize("width,sizes", [(64, (2, 3, 1, 4, 5, 2, 2)), (260, (9, 1, 64)), (1028, (33, 2, 2)), (4096, (257, 5)), (260, (513, 3)), (64, (518, 2))])
def test_boundaries_of_a_portion(ctx, tmp_path, width, sizes):
    cfg = synth.seq_config(width, 30, [L("wkv", 24, heads=1, dim=8), L("delta", None, heads=2, kv_heads=1, dim=8, vdim=4, conv=2), L("wkv", 40, heads=1, dim=8)], taps=4)
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=600, n_slots=1, max_context=700)
    toks, per = tokens_for(cfg, 2 * sum(sizes) if sum(sizes) < 99 else sum(sizes)), []
    want = seq_oracle.run(cfg, t, toks, per)
    assert err(run_portions(m, toks, sizes), want) < TOL["float32"]
    m.capture_layers()
    s, first = m.acquire(), sizes[0]
    m.forward(s, toks[:first])
    got = m.layers(first)
    m.close()
    for g, w in zip(got, per):
        assert err(g, w[:first]) < TOL["float32"]


# the gated part norms of several rows (k_seqmix.hip sq_gate_partnorm_rows_kernel): parts of one run of four numbers, that end inside a wave's first, second and third run, of its last ones; of more and of
# no whole fours (the other form), as are 8 rows and fewer; in bfloat16 with an inner size whose rounded rows alone are written and one whose product reads the others
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,dim,parts", [(8, 4, 8), (4, 64, 1), (5, 52, 1), (16, 32, 1), (33, 16, 1), (16, 64, 1), (17, 64, 1), (18, 9, 3), (16, 64, 8)])
def test_part_norms_of_several_rows(ctx, tmp_path, heads, dim, parts, dtype):
    cfg = synth.pupidra_config(64, 40, [synth.pupidra_layer("mamba2", synth.pupidra_mamba2(heads, dim, 16, 1, 4, parts))])
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype=dtype, max_batch=40, n_slots=1)
    toks = tokens_for(cfg, 60)
    assert err(run_portions(m, toks, (9, 8, 33, 10)), seq_oracle.run_pupidra(cfg, t, toks)) < TOL[dtype]
    m.close()


# a single token's queries, key and value made inside its attention (k_winattn.hip winattn_step_kernel, ROW): groups of more than sixteen heads without norms, whose blocks all append the row and of which one updates
# the block means; of twelve with norms of their own and kept rows (more of those, and norms over whole projections, have a launch in front: test_host_calls.py); a ring that wraps; a reader of another layer's keys and values; norms per head with queries that turn; means begun by a portion and finished by single tokens
@pytest.mark.parametrize("which", ["pool", "pool without norms", "keep", "keep 12", "head norms", "18 heads"])
@pytest.mark.parametrize("sizes", [(1,), (1, 1, 7, 1, 1, 1, 1)])
def test_a_token_that_appends_itself(ctx, tmp_path, which, sizes):
    V = 40
    if which.startswith("pool"):
        at = {"heads": 36, "kv_heads": 2, "dim": 32, "vdim": 32, "mask": {"size": 5, "pool": 3}, "rot": {"base": 100.0, "dims": 16}, "scale": 0.2}
        run, cfg = seq_oracle.run_parallel, synth.parallel_config(64, V, [synth.parallel_layer(None, at, {"heads": 1, "dim": 16, "vdim": 16, "tau": 4.0}, 1.0, 0.5)], taps=2)
    elif which.startswith("keep"):
        at = lambda size, keep, own=None: synth.pupidra_attention(24 if which == "keep 12" else 34, 2, 32, 32, 1.0, size, keep, own)
        run, cfg = seq_oracle.run_pupidra, synth.pupidra_config(64, V, [synth.pupidra_layer("attention", at(9, 20)), synth.pupidra_layer("attention", at(4, 7, 0))])
    else:
        run, cfg = seq_oracle.run_zusolix, synth.zusolix_config(64, V, [synth.zusolix_layer("attention", synth.zusolix_attention(36 if which == "18 heads" else 6, 2, 48, 32, 0.1, 5.0, (0.4, 7)), ff=64)])
    t = synth.seq_tensors(cfg)
    if which == "pool without norms": t = {n: v for n, v in t.items() if not n.endswith(("q.norm", "k.norm"))}  # (those over whole projections: a launch in front)
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, t)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=16, n_slots=1, max_context=100)
    toks = tokens_for(cfg, 50)
    assert err(run_portions(m, toks, sizes), run(cfg, t, toks)) < TOL["float32"]
    m.close()


# a single token's decay, its second product inside the scan (k_seqmix.hip sq_fold): ranks in whole eights and not, the longest there (32 in eights of bfloat16, else 24) and longer ones with a launch of its own
# (test_host_calls.py), in both formats; heads of few rows and of many; the next token's neighbour, behind a portion and behind single tokens
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rank", [1, 8, 13, 23, 24, 25, 32, 33, 64, 65])
def test_decay_of_a_single_token(ctx, tmp_path, rank, dtype):
    cfg = synth.seq_config(160, 40, [L("wkv", None, heads=2, dim=24), L("wkv", 24, heads=1, dim=250)], taps=2)
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 3, synth.seq_tensors(cfg, 3, rank))
    m = seqmodel.load_model(ctx, str(tmp_path), dtype=dtype, max_batch=16, n_slots=1)
    toks = tokens_for(cfg, 12)
    assert err(run_portions(m, toks, (1, 1, 5, 1, 1, 1)), seq_oracle.run(cfg, t, toks)) < TOL[dtype]
    m.close()


# the same decay in bfloat16 is a portion's: the vector in front of its second product is rounded in both.  w = exp(-exp(1024 a - 1020)) of an a that rounds from 0.995 to 255 / 256 for every token: 0.37, and 0.7 of one
# that is not rounded
@pytest.mark.parametrize("rank", [1, 8])
def test_decay_of_a_single_token_is_that_of_a_portion(ctx, tmp_path, rank):
    cfg = synth.seq_config(64, 40, [L("wkv", None, heads=2, dim=24)], taps=2)
    t = synth.seq_tensors(cfg, 3, rank)
    m = "l0.mix."
    t["embed"][:, 0] = 50.0  # a channel that is the same for every token, which the decay alone reads
    t["l0.norm1"][0] = t[m + "mu.w"][0] = 0.0
    t["l0.canon1"][0] = t["head"][:, 0] = 0.0
    for n in "rkvg": t[m + n][:, 0] = 0.0
    t[m + "w1"][:], t[m + "w2"][:], t[m + "w0"][:] = 0.0, 0.0, -1020.0
    t[m + "w1"][0, 0], t[m + "w2"][:, 0] = 0.38, 1024.0
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 3, t)
    model = seqmodel.load_model(ctx, str(tmp_path), dtype="bfloat16", max_batch=16, n_slots=1)
    toks = tokens_for(cfg, 12)
    assert err(run_portions(model, toks, (1,)), run_portions(model, toks, (12,))) < 0.02
    model.close()


# wkv and delta rule in chunks of 16 tokens (k_chunk.hip): portions that end inside, on and one behind a chunk's edge, fewer than 32 tokens between them (the scan), state row tiles that
# do not fill the four waves and more than they are, value columns that are no multiple of 16; decays from e^-20 a token to none at all
@pytest.mark.parametrize("sizes", [(31, 33), (32,), (47, 5, 49), (64, 17), (100,)])
def test_recurrences_in_chunks(made, sizes):
    cfg = synth.seq_config(64, 40, [L("wkv", None, heads=2, dim=16), L("delta", None, heads=4, kv_heads=2, dim=48, vdim=20, conv=3), L("wkv", None, heads=1, dim=80),
                                    L("delta", None, heads=1, kv_heads=1, dim=256, vdim=33, conv=2), L("delta", None, heads=3, kv_heads=1, dim=144, vdim=16, conv=1)], taps=2)
    t = synth.seq_tensors(cfg, 5)
    t["l0.mix.w0"], t["l2.mix.w0"] = np.linspace(-9, 3, 32, dtype=np.float32), np.linspace(3, -9, 80, dtype=np.float32)
    t["l1.mix.A_log"] = np.asarray([-9, -2, 1, 3], np.float32)
    t = {n: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(np.shape(a)) for n, a in t.items()}
    m, c, t = made("chunks", max_batch=100, cfg=cfg, tensors=t)
    toks = tokens_for(c, 230)
    assert err(run_portions(m, toks, sizes), seq_oracle.run(c, t, toks)) < TOL["float32"]


# the same scan without branches (k_chunk.hip chunk_scan_kernel, FULL: whole tiles for each of the four waves, one to four of them; heads in eights and not): two to nine chunks, so fewer than are
# requested ahead, one more, every number that the loop's three leave over, a last chunk of one, of fifteen and of sixteen tokens
@pytest.mark.parametrize("sizes", [(32, 33), (48, 63, 64), (65, 80, 81), (95, 96, 112), (127, 128, 130)])
def test_recurrences_in_whole_tiles(made, sizes):
    cfg = synth.seq_config(64, 40, [L("wkv", None, heads=8, dim=64), L("delta", None, heads=16, kv_heads=8, dim=64, vdim=32, conv=3), L("wkv", None, heads=1, dim=128),
                                    L("delta", None, heads=2, kv_heads=1, dim=192, vdim=16, conv=2), L("delta", None, heads=8, kv_heads=2, dim=128, vdim=48, conv=1), L("wkv", None, heads=2, dim=256),
                                    L("delta", None, heads=1, kv_heads=1, dim=256, vdim=64, conv=2)], taps=2)
    t = synth.seq_tensors(cfg, 5)
    t["l0.mix.w0"], t["l2.mix.w0"] = np.linspace(-9, 3, 512, dtype=np.float32), np.linspace(3, -9, 128, dtype=np.float32)
    t["l1.mix.A_log"] = np.linspace(-9, 3, 16, dtype=np.float32)
    t = {n: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(np.shape(a)) for n, a in t.items()}
    m, c, t = made("whole-tiles", max_batch=130, cfg=cfg, tensors=t)
    toks = tokens_for(c, sum(sizes) + 40)
    assert err(run_portions(m, toks, sizes), seq_oracle.run(c, t, toks)) < TOL["float32"]


# channels and heads that forget everything at once at some tokens and next to nothing at others: a token's log decay runs from nothing over e^30 .. e^45, where a running sum of them would
# swallow the ordinary decays behind it, to an overflow of fp32; the state that the next portion starts from is right too.  (32 tokens and more: chunks; 31 and fewer: the scan)
@pytest.mark.parametrize("sizes", [(32,), (47, 5, 49), (31, 33)])
def test_recurrences_in_chunks_that_forget_everything(made, sizes):
    cfg = synth.seq_config(64, 40, [L("wkv", None, heads=2, dim=32), L("delta", None, heads=4, kv_heads=2, dim=32, vdim=20, conv=2)], taps=2)
    t = synth.seq_tensors(cfg, 6)
    gain = np.tile(np.float32([1, 15, 30, 45, 60, 95, 0, 1]), 8)[:, None]  # z = w0 + gain times a number of about 0.6
    t["l0.mix.w2"] = t["l0.mix.w2"] * gain
    t["l0.mix.w0"] = np.tile(np.float32([0, 0, 0, 0, 0, 0, 92, 37]), 8)
    t["l1.mix.a"] = t["l1.mix.a"] * np.float32([[1], [30], [30], [1]])
    t["l1.mix.A_log"] = np.float32([1, 30, 37, 92])
    t = {n: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(np.shape(a)) for n, a in t.items()}
    m, c, t = made("forget", max_batch=64, cfg=cfg, tensors=t)
    toks = tokens_for(c, 150)
    with np.errstate(over="ignore"):
        want = seq_oracle.run(c, t, toks)
    assert err(run_portions(m, toks, sizes), want) < TOL["float32"]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T,N,K", [(1, 37, 50), (2, 64, 96), (3, 19, 7), (8, 130, 72), (9, 70, 33), (70, 129, 200), (200, 48, 48), (1, 16, 4096)])
def test_dense_matmul_any_shape(ctx, dtype, T, N, K):
    rng = np.random.default_rng(T * 1000 + N)
    w = rng.standard_normal((N, K), dtype=np.float32)
    x = rng.standard_normal((T, K), dtype=np.float32)
    from powerserve_amd.safetensors_io import f32_to_bf16_bits
    bits = f32_to_bf16_bits(w)
    rnd = lambda a: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(a.shape)
    import ctypes as C
    h = C.c_void_p()
    ctx.check(ctx.L.ps_hip_dense_upload(ctx.h, bits.ctypes.data_as(C.c_void_p), N, K, int(dtype == "float32"), C.byref(h)))
    dx, do = ctx.to_device(x), ctx.empty((T, N))
    ctx.check(ctx.L.ps_hip_dense_matmul(ctx.h, h, dx.ptr, T, do.ptr, 0.5))
    ctx.sync()
    xr = x if dtype == "float32" else rnd(x)
    want = 0.5 * (xr.astype(np.float64) @ rnd(w).astype(np.float64).T)
    assert np.abs(do.numpy() - want).max() < 1e-4 * max(1.0, np.abs(want).max())
    ctx.L.ps_hip_dense_free(ctx.h, h)
    dx.free(); do.free()


# a token at a time: boundaries and norms of one run per thread, a run and four numbers more, two runs, no multiple of four (the general kernels), one, two and four taps; the absorbed
# attention with one and two groups of value columns per wave, heads in and one beyond a tile of 16, windows of one tile, one key more and of two tiles, more than nine pieces of a key per wave
@pytest.mark.parametrize("width,taps,heads,rank,rot,window", [(64, 4, 1, 16, 16, 16), (4096, 1, 16, 64, 16, 17), (4100, 4, 17, 272, 16, 32), (4104, 1, 3, 512, 32, 5), (8192, 4, 2, 256, 336, 20),
                                                            (66, 4, 2, 48, 16, 7), (132, 2, 2, 512, 80, 18)])
def test_kernels_of_a_single_token(made, width, taps, heads, rank, rot, window):
    cfg = synth.seq_config(width, 40, [L("latent_attention", 24, heads=heads, dim=16, vdim=12, q_rank=20, kv_rank=rank, mask={"size": window}, scale=0.3, rot={"base": 100.0, "dims": 12},
                                         rot_dim=rot), L("wkv", None, heads=1, dim=20)], taps=taps)
    m, c, t = made(f"one{width}.{rank}", max_batch=16, cfg=cfg)
    toks = tokens_for(c, 45)
    assert err(run_portions(m, toks, (1,)), seq_oracle.run(c, t, toks)) < TOL["float32"]


# heads' norms and gates inside a token's output projection (k_dense.hip dn_stage_pre): heads of four numbers, of a wave's 256, one run of 2048 and less than one; sizes it does not take (no whole
# units, heads of 48 numbers); steps of one token that are asked for nothing, once and twice
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,dim,vdim", [(128, 4, 4), (2, 256, 256), (16, 128, 128), (1, 64, 512), (4, 16, 64), (16, 16, 48), (12, 32, 128)])
def test_norms_in_front_of_a_tokens_output_projection(made, heads, dim, vdim, dtype):
    layers = [L("delta", 24, heads=heads, kv_heads=1, dim=dim, vdim=vdim, conv=2)] + ([L("wkv", None, heads=heads, dim=dim)] if dim == vdim else [])
    cfg = synth.seq_config(64, 40, layers[:1] if dtype == "bfloat16" else layers, taps=4)
    m, c, t = made(f"pre{heads}.{dim}.{vdim}", dtype, cfg=cfg)
    toks = tokens_for(c, 24)
    want = seq_oracle.run(c, t, toks)
    assert err(run_portions(m, toks, (1,)), want) < TOL[dtype]
    s = m.acquire()
    for i in range(0, 24, 3):
        m.forward(s, toks[i:i + 1])
        assert err(m.forward(s, toks[i + 1:i + 2], [0, 0]), want[[i + 1, i + 1]]) < TOL[dtype]
        m.forward(s, toks[i + 2:i + 3], [0])
    m.release(s)


# a single token behind a window of very many keys (k_latent.hip latent_combine_kernel): as many tiles as it keeps the weights of, one more, and more than LDS has room for
@pytest.mark.parametrize("window", [262_128, 262_129, 652_000])
def test_latent_attention_of_a_very_long_window(ctx, tmp_path, window):
    cfg = synth.seq_config(64, 40, [L("latent_attention", None, heads=2, dim=16, vdim=16, q_rank=20, kv_rank=16, mask={"size": window}, scale=0.3, rot={"base": 100.0, "dims": 16}, rot_dim=16)],
                           taps=2)
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=4, n_slots=1, max_context=700_000)
    toks = tokens_for(cfg, 100)
    got = run_portions(m, toks, (1,))
    m.close()
    assert err(got, seq_oracle.run(cfg, t, toks)) < TOL["float32"]


# the wide mat-mul (k_dense.hip dense_mm_ring_kernel): one row more and less than its tiles of 64 and 128 tokens and outputs, one block of K and fewer blocks than stages,
# products split along K (few tiles, long K: also uneven shares), more tiles than the chip has CUs
@pytest.mark.parametrize("dtype", list(FORMS))
@pytest.mark.parametrize("T,N,K", [(9, 1, 64), (63, 127, 128), (64, 128, 192), (65, 129, 256), (127, 63, 320), (128, 65, 576), (129, 200, 64), (300, 130, 1088), (16, 8, 4096), (40, 100, 4160),
                                   (200, 256, 2240), (520, 2100, 128),
                                   # many tiles of few blocks of K (every form by its name: test_dense_matmul_of_every_tile)
                                   (2047, 2100, 64), (2049, 2305, 64), (1999, 3001, 192), (1030, 4100, 320), (1793, 2304, 128), (300, 20004, 64)])
def test_dense_matmul_wide(ctx, dtype, T, N, K):
    import ctypes as C
    rng = np.random.default_rng(T * 1000 + N)
    bits = f32_to_bf16_bits(rng.standard_normal((N, K), dtype=np.float32))
    rnd = lambda a: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(a.shape)
    x = rng.standard_normal((T, K), dtype=np.float32)
    w = (bits.astype(np.uint32) << 16).view(np.float32).reshape(N, K)
    h = C.c_void_p()
    ctx.check(ctx.L.ps_hip_dense_upload(ctx.h, bits.ctypes.data_as(C.c_void_p), N, K, FORMS[dtype], C.byref(h)))
    assert ctx.L.ps_hip_dense_form(h) == FORMS[dtype]
    dx, do = ctx.to_device(x), ctx.to_device(np.full((T + 1, N), np.float32(7.0)))
    ctx.check(ctx.L.ps_hip_dense_matmul(ctx.h, h, dx.ptr, T, do.ptr, 1.0))
    got = do.numpy()
    a = (rnd(x) if dtype == "bfloat16" else x).astype(np.float64)
    # fp32 sums of K products, in any order: at most K roundings of 2^-24, each relative to a partial sum of at most sum |a w|
    bound = K * 2.0 ** -24 * (np.abs(a) @ np.abs(w.astype(np.float64)).T)
    assert np.all(np.abs(got[:T] - a @ w.astype(np.float64).T) <= bound)
    assert np.all(got[T] == 7.0)  # nothing behind the last row
    ctx.L.ps_hip_dense_free(ctx.h, h)
    dx.free(); do.free()


# the four-tap filter (k_seqmix.hip sq_conv4_kernel) in portions of one to nine tokens (its threads take four; the tail from old and new tokens) and the norms around it with one, two and four
# runs per thread, a run and four channels more, and in the general kernels (66: no multiple of four)
@pytest.mark.parametrize("width", [64, 66, 1024, 1028, 2052, 8192])
@pytest.mark.parametrize("sizes", [(2,), (3, 1), (4, 2, 1), (5, 9, 8)])
def test_filters_and_norms_of_portions(made, width, sizes):
    cfg = synth.seq_config(width, 40, [L("delta", 24, heads=2, kv_heads=1, dim=12, vdim=20, conv=4), L("delta", None, heads=2, kv_heads=2, dim=16, vdim=8, conv=4)], taps=4)
    m, c, t = made(f"four{width}", max_batch=16, cfg=cfg)
    toks = tokens_for(c, 37)
    assert err(run_portions(m, toks, sizes), seq_oracle.run(c, t, toks)) < TOL["float32"]


# the four token-shift products of a layer in one launch: columns that are whole tiles of 128 (the wide mat-mul; a tile's matrix changes with it) and that are not (one by one), a single token
# (its state vector 16-byte aligned and not: 20 channels of another layer in front), two to eight tokens (one by one), a portion split along K
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,heads,dim", [(64, 2, 64), (64, 3, 32), (72, 1, 128), (576, 2, 192), (1024, 4, 32), (66, 2, 20)])
def test_four_mixes_together(made, width, heads, dim, dtype):
    wkv = L("wkv", None, heads=heads, dim=dim)
    # (bfloat16: one layer, whose own roundings the tolerance is for; a recurrence over a recurrence carries them on)
    cfg = synth.seq_config(width, 40, [wkv] if dtype == "bfloat16" else [wkv, L("latent_attention", 24, heads=1, dim=8, vdim=12, q_rank=9, kv_rank=11, mask={"size": 3}, scale=1.0,
                                                                                rot={"base": 100.0, "dims": 2}, rot_dim=6), wkv], taps=2)
    m, c, t = made(f"mixes{width}.{heads}", dtype, max_batch=64, cfg=cfg)
    toks = tokens_for(c, 60)
    want = seq_oracle.run(c, t, toks)
    for sizes in ((1,), (5, 9, 2, 44)):
        e = err(run_portions(m, toks, sizes), want)
        assert e < TOL[dtype], (sizes, e)


# all four mixes of a row by one thread (k_dense.hip dense_pack_kernel, 512 rows of 1024 and more), in a portion that begins a sequence and one that does not
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_four_mixes_of_many_rows(ctx, tmp_path, dtype):
    cfg = synth.seq_config(1024, 40, [L("wkv", None, heads=4, dim=32)], taps=2)
    synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype=dtype, max_batch=520, n_slots=1, max_context=1100)
    toks = tokens_for(cfg, 1030)
    got = run_portions(m, toks, (520, 510))
    m.set_mode(2)  # the tiled mat-mul, which mixes where it reads
    want = run_portions(m, toks, (520, 510))
    m.close()
    # fp32: a few ulps of fp32 sums; bf16: a rounding now and then goes the other way.  A mix that is not its own: ~1
    assert err(got, want) < (TOL["float32"] if dtype == "float32" else 0.03)


# bf16 rows handed from one kernel to the wide mat-mul behind it (inputs of more than 256 numbers, whole blocks of 64): filter -> projection, head norm -> projection, first -> second product;
# beside them a projection that does not take them (260 is no multiple of 64), portions below and above the sizes that hand on, and what an earlier layer or portion left behind
@pytest.mark.parametrize("sizes", [(9, 8, 64), (33, 1), (64,)])
def test_bf16_rows_handed_on(made, sizes):
    cfg = synth.seq_config(320, 50, [L("wkv", 576, heads=5, dim=64), L("delta", 260, heads=6, kv_heads=3, dim=32, vdim=64, conv=4),
                                     L("latent_attention", 320, heads=5, dim=64, vdim=64, q_rank=64, kv_rank=64, mask={"size": 30}, scale=0.1, rot={"base": 500.0, "dims": 16}, rot_dim=16),
                                     L("delta", None, heads=2, kv_heads=2, dim=16, vdim=130, conv=4)], taps=4)
    m, c, t = made("handed", "bfloat16", max_batch=64, cfg=cfg)
    toks = tokens_for(c, 150)
    want, got = seq_oracle.run(c, t, toks), run_portions(m, toks, sizes)
    m.set_mode(2)  # the tiled mat-mul, which reads and rounds every operand itself
    plain = run_portions(m, toks, sizes)
    m.set_mode(0)
    # both round the same numbers; their fp32 sums differ in order, so a rounding behind them may go the other way: an error of the same origin and size.  A row that is not its own: ~1
    assert err(got, want) < 1.5 * err(plain, want) < 0.3


# fp32 products on the bf16 instruction (k_dense.hip dn_ring_take, three lines of the operand): numbers that round to infinity in bf16, infinite and NaN operands and weights, numbers of every size --
# finite rows and columns beside them as exact as ever, the others infinite or NaN as fp32 arithmetic has them
@pytest.mark.parametrize("T,N,K", [(16, 24, 64), (70, 130, 192), (700, 5000, 64)])
@pytest.mark.parametrize("odd_weights", [False, True])
@pytest.mark.parametrize("dtype", ["float32", "float32 lines"])
def test_float32_products_of_odd_numbers(ctx, T, N, K, odd_weights, dtype):
    import ctypes as C
    rng = np.random.default_rng(T)
    w = rng.standard_normal((N, K), dtype=np.float32)
    if odd_weights:
        w[3, 5], w[7, 1] = np.inf, np.nan
    bits = f32_to_bf16_bits(w)
    w = (bits.astype(np.uint32) << 16).view(np.float32).reshape(N, K)
    x = rng.standard_normal((T, K), dtype=np.float32)
    x[1] *= np.float32(10.0) ** rng.integers(-30, 30, K).astype(np.float32)
    x[2], x[2, 9] = 0, np.float32(3.4028e38)  # (the next bf16 is infinity)
    x[4, 0], x[5, 3] = np.inf, np.nan
    x[6] = 1  # (its lower lines are zeros)
    h = C.c_void_p()
    ctx.check(ctx.L.ps_hip_dense_upload(ctx.h, bits.ctypes.data_as(C.c_void_p), N, K, FORMS[dtype], C.byref(h)))
    assert ctx.L.ps_hip_dense_form(h) == (hip.DENSE_F32 if odd_weights else FORMS[dtype])
    dx, do = ctx.to_device(x), ctx.empty((T, N))
    ctx.check(ctx.L.ps_hip_dense_matmul(ctx.h, h, dx.ptr, T, do.ptr, 2.0 ** -8))
    got = do.numpy()
    with np.errstate(all="ignore"):
        want = (x.astype(np.float64) @ w.astype(np.float64).T) * 2.0 ** -8
        bound = (K + 2) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T) * 2.0 ** -8
        over, beyond = (np.abs(want) * 2.0 ** 8 > v for v in (3.4e38, 3.41e38))  # (fp32's largest number is 3.4028e38: sums near it may or may not end at infinity, sums beyond it do)
    fine = np.isfinite(want) & ~over
    assert np.all(np.abs(got[fine] - want[fine]) <= bound[fine])
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~np.isfinite(want) & ~np.isnan(want)], want[~np.isfinite(want) & ~np.isnan(want)].astype(np.float32))
    assert np.all(np.isinf(got[beyond & np.isfinite(want)]))
    ctx.L.ps_hip_dense_free(ctx.h, h)
    dx.free(); do.free()


# a float32 model in either form of its matrices: four mixes, a feed-forward and a latent's window large enough (what is small runs on the fp32 instruction in both: psk_dense_args small_f32),
# experts; a joint projection of two mixers; portions and single tokens
@pytest.mark.parametrize("dtype", ["float32", "float32 lines"])
@pytest.mark.parametrize("which", ["mixes", "experts", "joint"])
def test_float32_models_in_either_form(ctx, tmp_path, which, dtype):
    V = 40
    if which == "mixes":
        run, cfg = seq_oracle.run, synth.seq_config(128, V, [L("wkv", 192, heads=4, dim=32), L("latent_attention", 8256, heads=16, dim=128, vdim=128, q_rank=64, kv_rank=320, mask={"size": 33}, scale=0.1,
                                                                                             rot={"base": 100.0, "dims": 8}, rot_dim=16), L("delta", 64, heads=4, kv_heads=2, dim=32, vdim=32, conv=3)], taps=2)
    elif which == "experts":
        run, cfg = seq_oracle.run_pupidra, synth.pupidra_config(128, V, [synth.pupidra_layer("attention", synth.pupidra_attention(2, 1, 64, 64, 0.3, 9, 2), moe=(5, 2, 128, 1.7), shared=64)])
    else:
        run, cfg = seq_oracle.run_parallel, synth.parallel_config(512, V, [synth.parallel_layer(128, {"heads": 8, "kv_heads": 2, "dim": 64, "vdim": 64, "mask": {"size": 33, "pool": 3},
                                                                  "rot": {"base": 100.0, "dims": 16}, "scale": 0.2}, {"heads": 8, "dim": 64, "vdim": 64, "tau": 4.0}, 1.0, 0.5)], taps=2)
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=300, n_slots=1, max_context=700, f32_form=FORMS[dtype])
    assert {ctx.L.ps_hip_dense_form(w) for w in m._up.mats} == {FORMS[dtype]}
    toks = tokens_for(cfg, 350)
    assert err(run_portions(m, toks, (300, 1, 5, 44)), run(cfg, t, toks)) < TOL["float32"]
    m.close()


# a small matrix and few rows of a float32 model: on either side of the line between the fp32 instruction and three lines (k_dense.hip dn_wide), by rows (1024 x 1024: 256; 1024 x 4096: 64) and by the matrix (1024 x 4160)
@pytest.mark.parametrize("ff,sizes", [(1024, (256, 5)), (1024, (257, 4)), (4096, (64, 65)), (4160, (64, 9))])
def test_small_float32_products(made, ff, sizes):
    cfg = synth.seq_config(1024, 40, [L("delta", ff, heads=2, kv_heads=1, dim=16, vdim=16, conv=2)], taps=2)
    m, c, t = made(f"small-f32.{ff}", max_batch=260, cfg=cfg)
    toks = tokens_for(c, 261)
    assert {m.ctx.L.ps_hip_dense_form(w) for w in m._up.mats} == {hip.DENSE_F32_LINES}
    assert err(run_portions(m, toks, sizes), seq_oracle.run(c, t, toks)) < TOL["float32"]


# wide tiles behind an epilogue (by their names: test_every_tile_behind_an_epilogue): an activation whose rounded rows the second product reads, pairs, the four mixes of a token shift, the slots of
# experts (tiles that end inside an expert, an expert without slots) with a factor per row
@pytest.mark.parametrize("which", ["xielu", "pairs", "experts", "mixes"])
def test_large_tiles_behind_an_epilogue(ctx, tmp_path, which):
    V = 30
    if which == "experts":
        cfg = synth.pupidra_config(64, V, [synth.pupidra_layer("attention", synth.pupidra_attention(2, 1, 16, 16, 0.3, 9, 2), moe=(5, 2, 6144, 1.7), shared=8)])
    elif which == "mixes":
        cfg = synth.seq_config(64, V, [L("wkv", None, heads=16, dim=128)], taps=2)
    elif which == "pairs":
        cfg = synth.pokatar_config(64, V, [synth.pokatar_layer("attention", synth.pokatar_attention(2, 1, 16, 16, 0.3), 4096)])
    else:
        cfg = synth.seq_config(64, V, [L("delta", 8192, heads=2, kv_heads=1, dim=16, vdim=16, conv=2)], taps=2)
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="bfloat16", max_batch=640, n_slots=1, max_context=700)
    toks = tokens_for(cfg, 600)
    got = run_portions(m, toks, (600,))
    m.set_mode(2)  # the tiled mat-mul
    plain = run_portions(m, toks, (600,))
    m.close()
    # both round the same numbers; their fp32 sums differ in order, so a rounding behind them may go the other way (2^-9 of a number, a few numbers of a row).  A row that is not its own: ~1
    assert err(got, plain) < 0.03


# matrices counted by the lanes of a wave (k_dense.hip dn_ring_rows): as many experts as lanes, one and two more, three waves full; few tokens, most of whose experts have no slot, and portions in which
# they have from none to many; products whole and, behind a short inner size, in parts of K
@pytest.mark.parametrize("dtype", ["float32", "float32 lines", "bfloat16"])
@pytest.mark.parametrize("experts,ff", [(64, 128), (65, 64), (66, 192), (192, 64), (70, 1152)])
def test_more_experts_than_lanes(ctx, tmp_path, experts, ff, dtype):
    cfg = synth.pupidra_config(128, 40, [synth.pupidra_layer("attention", synth.pupidra_attention(2, 1, 16, 16, 0.3, 9, 2), moe=(experts, 3, ff, 1.7), shared=8)])
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype=dtype.split()[0], max_batch=300, n_slots=1, max_context=400, f32_form=None if dtype == "bfloat16" else FORMS[dtype])
    toks = tokens_for(cfg, 320)
    got = run_portions(m, toks, (9, 300, 11))
    if dtype == "bfloat16":  # (a near tie may be routed the other way behind 16 bits: against the tiled mat-mul)
        m.set_mode(2)
        want = run_portions(m, toks, (9, 300, 11))
    else:
        want = seq_oracle.run_pupidra(cfg, t, toks)
    m.close()
    assert err(got, want) < (0.03 if dtype == "bfloat16" else TOL["float32"])


# the same for the tiles of 256 columns at each of their heights, and for 192 x 128 whole and in parts (wide_tiles.py; which kernel runs: test_host_calls.py)
@pytest.mark.parametrize("which,dtype,size,tokens,width", [(which, dtype, *case[:3]) for (which, dtype), cases in wide_tiles.EPILOGUES.items() for case in cases])
def test_every_tile_behind_an_epilogue(ctx, tmp_path, which, dtype, size, tokens, width):
    cfg = wide_tiles.layers(synth, which, size, width)
    synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype=dtype, max_batch=tokens, n_slots=1, max_context=tokens + 100, f32_form=FORMS["float32 lines"] if dtype == "float32" else None)
    toks = tokens_for(cfg, tokens)
    got = run_portions(m, toks, (tokens,))
    m.set_mode(2)  # the tiled mat-mul
    plain = run_portions(m, toks, (tokens,))
    m.close()
    assert err(got, plain) < (0.03 if dtype == "bfloat16" else TOL["float32"])  # (bf16: as above)


# xIELU behind a wide product (k_dense.hip dn_xielu): arguments from 2^-20 to beyond -64, where its exponent is held; rows of the first product scaled up and the second's columns down, so
# that every scale counts alike in the result
def test_activation_of_any_size(made):
    cfg = synth.seq_config(64, 40, [L("wkv", 128, heads=2, dim=16)], taps=2)
    t = synth.seq_tensors(cfg, 11)
    scale = np.exp2(np.linspace(-20, 9, 128, dtype=np.float32))
    t["l0.mlp.up"] = t["l0.mlp.up"] * scale[:, None]
    t["l0.mlp.down"] = t["l0.mlp.down"] / np.maximum(scale, scale * scale)
    t = {n: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(np.shape(a)) for n, a in t.items()}
    m, c, t = made("xielu", max_batch=64, cfg=cfg, tensors=t)
    toks = tokens_for(c, 100)
    assert err(run_portions(m, toks, (64, 36)), seq_oracle.run(c, t, toks)) < TOL["float32"]


# attention of many rows with its operands split into three bf16 numbers (k_splitattn.hip: two blocks of 128 rows of 64 heads and more): keys of 192 and 128 numbers, windows that end inside blocks of
# 32 keys and inside a portion, with and without kept first tokens (fewer and more than a block), means of blocks, distance slopes, a reader of another layer's keys, gates, temperatures and sinks,
# a soft cap, rotated queries of both pairings, key / value groups; a ring that has wrapped; portions of fewer rows (the fp32 instruction) in between; one row of the last block of 128
@pytest.mark.parametrize("which", ["latent", "latent direct", "keep", "pool", "softcap"])
def test_attention_of_many_rows(ctx, tmp_path, which):
    V, sizes = 40, (200, 1, 129, 140)
    if which == "latent":
        run, cfg = seq_oracle.run, synth.seq_config(64, V, [L("latent_attention", None, heads=64, dim=128, vdim=128, q_rank=40, kv_rank=64, mask={"size": 77}, scale=0.09,
                                                              rot={"base": 500.0, "dims": 48}, rot_dim=64)], taps=2)
    elif which == "latent direct":
        run, cfg = seq_oracle.run_pupidra, synth.pupidra_config(64, V, [synth.pupidra_layer("latent_attention", synth.pupidra_latent(64, 96, 32, 128, 32, 0.1, 1e4))])
    elif which == "keep":
        at = lambda size, keep, own=None: synth.pupidra_attention(64, 2, 128, 128, 1.0, size, keep, own)
        run, cfg = seq_oracle.run_pupidra, synth.pupidra_config(64, V, [synth.pupidra_layer("attention", at(150, 40)), synth.pupidra_layer("attention", at(31, 5, 0))])
    elif which == "pool":
        at = {"heads": 64, "kv_heads": 4, "dim": 128, "vdim": 128, "mask": {"size": 33, "pool": 3}, "rot": {"base": 100.0, "dims": 64}, "scale": 0.1}
        run, cfg = seq_oracle.run_parallel, synth.parallel_config(64, V, [synth.parallel_layer(None, at, {"heads": 1, "dim": 16, "vdim": 16, "tau": 4.0}, 1.0, 0.5)], taps=2)
    else:
        run, cfg = seq_oracle.run_zusolix, synth.zusolix_config(64, V, [synth.zusolix_layer("attention", synth.zusolix_attention(64, 8, 128, 128, 0.1, 5.0, (0.4, 7)), ff=64)])
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=200, n_slots=1, max_context=500)
    toks = tokens_for(cfg, sum(sizes))
    want, got = run(cfg, t, toks), run_portions(m, toks, sizes)
    m.set_mode(2)  # the plain kernels
    plain = run_portions(m, toks, sizes)
    m.close()
    assert err(got, want) < min(TOL["float32"], 2 * err(plain, want) + 2e-6)


# the same with rows whose keys several work-groups share (k_splitattn.hip split_join_kernel; two parts, in the second portion): parts in which some rows, or all, see no key; kept first tokens and means of
# blocks in parts of their own; the last rows of a tile missing; sinks, gates, a soft cap and slopes behind the sum.  "latent odd": whole tiles, queries turned beforehand, in rows that no 16-byte load
# fits (81 gates behind them)
@pytest.mark.parametrize("which", ["latent", "latent odd", "keep", "pool", "softcap"])
def test_attention_of_many_rows_in_parts(ctx, tmp_path, which):
    V, sizes = 40, (260, 140)
    if which == "latent":
        run, cfg = seq_oracle.run, synth.seq_config(64, V, [L("latent_attention", None, heads=64, dim=128, vdim=128, q_rank=40, kv_rank=64, mask={"size": 390}, scale=0.09,
                                                              rot={"base": 500.0, "dims": 48}, rot_dim=64)], taps=2)
    elif which == "latent odd":
        run, cfg = seq_oracle.run_pupidra, synth.pupidra_config(64, V, [synth.pupidra_layer("latent_attention", synth.pupidra_latent(81, 96, 32, 128, 32, 0.1, 1e4))])
    elif which == "keep":
        at = lambda size, keep, own=None: synth.pupidra_attention(64, 2, 128, 128, 1.0, size, keep, own)
        run, cfg = seq_oracle.run_pupidra, synth.pupidra_config(64, V, [synth.pupidra_layer("attention", at(150, 200)), synth.pupidra_layer("attention", at(310, 5, 0))])
    elif which == "pool":
        at = {"heads": 64, "kv_heads": 4, "dim": 128, "vdim": 128, "mask": {"size": 33, "pool": 2}, "rot": {"base": 100.0, "dims": 64}, "scale": 0.1}
        run, cfg = seq_oracle.run_parallel, synth.parallel_config(64, V, [synth.parallel_layer(None, at, {"heads": 1, "dim": 16, "vdim": 16, "tau": 4.0}, 1.0, 0.5)], taps=2)
    else:
        run, cfg = seq_oracle.run_zusolix, synth.zusolix_config(64, V, [synth.zusolix_layer("attention", synth.zusolix_attention(64, 8, 128, 128, 0.1, 5.0, (0.4, 7)), ff=64)])
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=100, n_slots=1, max_context=500)
    toks = tokens_for(cfg, sum(sizes))
    want, got = run(cfg, t, toks), run_portions(m, toks, sizes)
    m.set_mode(2)  # the plain kernels
    plain = run_portions(m, toks, sizes)
    m.close()
    assert err(got, want) < min(TOL["float32"], 2 * err(plain, want) + 2e-6)


# tiles of one, two and three parts in one launch (260 tokens of 41 heads: 4, 8 and 9 blocks), then two of three parts each (the launches: test_host_calls.py); queries turned beforehand in rows that no
# 16-byte load fits (41 gates behind them), a soft cap and gates
@pytest.mark.parametrize("which", ["latent odd", "softcap"])
def test_attention_of_tiles_in_one_to_three_parts(ctx, tmp_path, which):
    V, sizes = 40, (260, 200)
    if which == "latent odd":
        run, cfg = seq_oracle.run_pupidra, synth.pupidra_config(64, V, [synth.pupidra_layer("latent_attention", synth.pupidra_latent(41, 96, 32, 128, 32, 0.1, 1e4))])
    else:
        run, cfg = seq_oracle.run_zusolix, synth.zusolix_config(64, V, [synth.zusolix_layer("attention", synth.zusolix_attention(41, 1, 128, 128, 0.1, 5.0, (0.4, 7)), ff=64)])
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=260, n_slots=1, max_context=500)
    toks = tokens_for(cfg, sum(sizes))
    want, got = run(cfg, t, toks), run_portions(m, toks, sizes)
    m.set_mode(2)  # the plain kernels
    plain = run_portions(m, toks, sizes)
    m.close()
    assert err(got, want) < min(TOL["float32"], 2 * err(plain, want) + 2e-6)


# the same attention with an infinite key, value or query of one token (64 heads of 150 and 140 rows: k_splitattn.hip): a score of -inf is a weight of nothing, an infinite value makes the rows that see
# it infinite (not NaN), and rows that do not see the token -- those in front of it in the same 16 rows and 32 keys too -- are what they are without it
@pytest.mark.parametrize("what", ["k", "v", "q"])
def test_attention_of_many_rows_with_infinite_numbers(ctx, tmp_path, what):
    cfg = synth.zusolix_config(64, 40, [synth.zusolix_layer("attention", synth.zusolix_attention(64, 8, 128, 128, 0.1))])
    t = {n: a.copy() for n, a in synth.seq_tensors(cfg, 0).items()}
    t["embed"][:, 3] = 0
    t["embed"][7, 3] = 30  # token 7 alone has channel 3; of the norm's 8 = sqrt(64) it gets most
    t["l0.norm1"][3] = 1
    heads, row = range(24, 32), (25 if what == "q" else 3) * 128 + 5  # channel 5 of key / value head 3, which these heads read, or of head 25's query
    for h in heads:
        t["l0.mix.q"][h * 128 + 5], t["l0.mix.q.b"][h * 128 + 5] = 0, -5  # (a negative score with an infinite key)
        t["l0.mix.o"][:, h * 128 + 5] = np.abs(t["l0.mix.o"][:, h * 128 + 5]) + 0.01
    t["l0.mix." + what][row], t["l0.mix." + what + ".b"][row] = 0, 0
    t["l0.mix." + what][row, 3] = 3e38
    t = {n: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(np.shape(a)) for n, a in t.items()}
    synth.write_seq_model_dir(str(tmp_path), cfg, 0, t)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=200, n_slots=1, max_context=500)
    toks = tokens_for(cfg, 290)
    toks[toks == 7] = 8
    toks[[20, 187]] = 7
    per = []
    seq_oracle.run_zusolix(cfg, t, toks, per)
    m.capture_layers()
    s, got = m.acquire(), []
    for part in (toks[:150], toks[150:]):
        m.forward(s, part)
        got.append(m.layers(part.size)[-1].copy())
    m.close()
    got, want, at = np.concatenate(got), per[-1], np.arange(290)
    fine = {"k": at >= 0, "v": at < 20, "q": toks != 7}[what]
    assert np.all(np.isfinite(got[fine]))
    assert np.abs(got[fine] - want[fine]).max() < TOL["float32"] * np.sqrt(np.mean(want[fine] ** 2))
    if what == "v":
        assert np.all(np.isinf(got[~fine])) and np.array_equal(np.sign(got[~fine]), np.sign(want[~fine]))


# results without an epilogue (k_dense.hip dense_mm_ring_kernel): columns in fours, stored from the registers, the last four of a tile, one four and three fours into the next one; no fours
# (through LDS); split along K, where the sums are stored in fours or one by one
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T,N,K", [(9, 4, 64), (65, 60, 128), (130, 132, 192), (513, 2060, 128), (130, 134, 192), (33, 36, 4160), (31, 68, 4096), (40, 102, 4160)])
def test_dense_matmul_stored_in_fours(ctx, dtype, T, N, K):
    test_dense_matmul_wide(ctx, dtype, T, N, K)


# the same with an activation, a bias or a sum behind rows that no 16-byte store fits (k_dense.hip dn_put4<true>), in the product and in the sums of its splits
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,ff", [(64, 130), (128, 258), (4160, 67)])
def test_odd_rows_behind_an_epilogue(made, dtype, width, ff):
    cfg = synth.seq_config(width, 50, [L("wkv", ff, heads=2, dim=16)], taps=2)
    m, cfg, t = made("odd-%d" % width, dtype, max_batch=64, cfg=cfg)
    toks = tokens_for(cfg, 75, seed=ff)
    assert err(run_portions(m, toks, [64, 11]), seq_oracle.run(cfg, t, toks)) < TOL[dtype]


# few blocks of K: a row, a column and four columns more and less than a tile of 128 and 192 rows x 256 columns and of 192 x 128, no fours; columns of tiles that are no multiple of a panel or of the XCDs
@pytest.mark.parametrize("dtype", list(FORMS))
@pytest.mark.parametrize("T,N,K", [(1153, 6148, 64), (641, 8196, 64), (1345, 3076, 64), (640, 8192, 128), (385, 14340, 320), (1345, 6145, 192), (2047, 4100, 192), (1025, 8200, 192), (1537, 2049, 192),
                                   (1345, 3077, 256), (193, 14340, 64), (577, 2052, 2112), (1345, 3076, 1088), (961, 4101, 1088)])
def test_dense_matmul_of_other_tile_heights(ctx, dtype, T, N, K):
    test_dense_matmul_wide(ctx, dtype, T, N, K)


# every tile of the wide mat-mul, whole and in parts of K (wide_tiles.py; which kernel runs: test_host_calls.py)
@pytest.mark.parametrize("dtype,T,N,K", [(dtype, T, N, K) for (dtype, _, _), sizes in wide_tiles.PRODUCTS.items() for T, N, K, _ in sizes])
def test_dense_matmul_of_every_tile(ctx, dtype, T, N, K):
    test_dense_matmul_wide(ctx, dtype, T, N, K)


# K up to 32 (k_dense.hip dense_mm_few_kernel): one below, at and above its two widths (33: the tiled kernel), one token and one column more and less than a work-group's
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T,N,K", [(9, 1, 1), (15, 255, 7), (16, 256, 8), (17, 257, 9), (33, 70, 31), (31, 513, 32), (40, 65, 33)])
def test_dense_matmul_of_a_short_inner_size(ctx, dtype, T, N, K):
    test_dense_matmul_wide(ctx, dtype, T, N, K)


# K a multiple of 128 up to 1024 and few tiles (k_dense.hip dense_mm_narrow_kernel): every number of steps per wave, a row and a column more and less than a tile, as many tiles as CUs and more
# (the ring), one step more of K (the ring)
@pytest.mark.parametrize("dtype", list(FORMS))
@pytest.mark.parametrize("T,N,K", [(9, 1, 128), (33, 31, 256), (31, 33, 384), (32, 64, 512), (65, 40, 640), (12, 100, 768), (40, 65, 896), (64, 129, 1024), (256, 1024, 512), (257, 1024, 512), (9, 70, 1152)])
def test_dense_matmul_of_few_tiles(ctx, dtype, T, N, K):
    test_dense_matmul_wide(ctx, dtype, T, N, K)


# two to eight tokens on the wide mat-mul (ps_seq.h PSD_FEW): the narrow tiles, the ring with and without a split along K, and the mat-vec where K is no whole 128 bytes (the same bound)
@pytest.mark.parametrize("dtype", list(FORMS))
@pytest.mark.parametrize("T,N,K", [(2, 1, 64), (3, 33, 128), (4, 129, 1024), (5, 70, 4160), (8, 2100, 192), (7, 65, 2048), (2, 300, 72), (8, 40, 1056)])
def test_dense_matmul_of_a_few_tokens(ctx, dtype, T, N, K):
    test_dense_matmul_wide(ctx, dtype, T, N, K)


# both sides of the lines between the mat-vec and the wide mat-mul for two to four tokens (k_dense.hip dn_few_first)
@pytest.mark.parametrize("dtype", list(FORMS))
@pytest.mark.parametrize("T,N,K", [(2, 70, 2048), (2, 70, 2112), (2, 33, 3072), (2, 33, 3136), (2, 600, 2432), (2, 607, 2432), (3, 256, 64), (4, 255, 64), (5, 300, 64)])
def test_dense_matmul_on_either_side_of_its_lines(ctx, dtype, T, N, K):
    test_dense_matmul_wide(ctx, dtype, T, N, K)


# one token (k_dense.hip dense_mv1_kernel): a row of less than one unit of its stream (512 numbers, fp32: 256), of exactly one, of one and a bit; fewer and more units per wave than are in flight;
# one row, rows that are no multiple of the waves', more rows than waves and more than 64 of them per wave; the longest row that is taken, and one more, which the general kernel does
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("N,K", [(1, 8), (7, 248), (9, 256), (65, 264), (8, 504), (63, 512), (66, 520), (1, 4096), (5, 4104), (4097, 64), (300001, 16), (12289, 520), (17, 32768), (17, 32776)])
def test_dense_matvec_in_one_stream(ctx, dtype, N, K):
    import ctypes as C
    rng = np.random.default_rng(N + K)
    bits = f32_to_bf16_bits(rng.standard_normal((N, K), dtype=np.float32))
    x = rng.standard_normal((1, K), dtype=np.float32)
    w = (bits.astype(np.uint32) << 16).view(np.float32).reshape(N, K)
    h = C.c_void_p()
    ctx.check(ctx.L.ps_hip_dense_upload(ctx.h, bits.ctypes.data_as(C.c_void_p), N, K, int(dtype == "float32"), C.byref(h)))
    dx, do = ctx.to_device(x), ctx.to_device(np.full((2, N), np.float32(7.0)))
    ctx.check(ctx.L.ps_hip_dense_matmul(ctx.h, h, dx.ptr, 1, do.ptr, 1.0))
    got = do.numpy()
    a = (x if dtype == "float32" else (f32_to_bf16_bits(x).astype(np.uint32) << 16).view(np.float32).reshape(x.shape)).astype(np.float64)
    # fp32 sums of K products, in any order: at most K roundings of 2^-24, each relative to a partial sum of at most sum |a w|
    assert np.all(np.abs(got[0] - (w.astype(np.float64) @ a[0])) <= K * 2.0 ** -24 * (np.abs(w).astype(np.float64) @ np.abs(a[0])))
    assert np.all(got[1] == 7.0)  # nothing behind the last row
    ctx.L.ps_hip_dense_free(ctx.h, h)
    dx.free(); do.free()


# a weight that is infinite stays infinite in its row's result, and in no other, wherever the row ends in the stream's last unit (one token) and with more tokens
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("N,K", [(5, 8), (9, 264), (12, 520), (33, 4104), (9, 512)])
def test_dense_matvec_with_an_infinite_weight(ctx, dtype, N, K, T):
    import ctypes as C
    rng = np.random.default_rng(N + K)
    bits = f32_to_bf16_bits(rng.standard_normal((N, K), dtype=np.float32))
    bits[3, 0], bits[1, K - 1] = 0x7F80, 0xFF80  # the first number of a row (what a lane beyond the row's end may be tempted to read), and the last
    x = rng.uniform(0.5, 1.0, (T, K)).astype(np.float32)
    w = (bits.astype(np.uint32) << 16).view(np.float32).reshape(N, K)
    h = C.c_void_p()
    ctx.check(ctx.L.ps_hip_dense_upload(ctx.h, bits.ctypes.data_as(C.c_void_p), N, K, int(dtype == "float32"), C.byref(h)))
    dx, do = ctx.to_device(x), ctx.to_device(np.zeros((T, N), np.float32))
    ctx.check(ctx.L.ps_hip_dense_matmul(ctx.h, h, dx.ptr, T, do.ptr, 1.0))
    got = do.numpy()
    assert np.all(got[:, 3] == np.inf) and np.all(got[:, 1] == -np.inf)
    finite = [n for n in range(N) if n not in (1, 3)]
    want = (x if dtype == "float32" else (f32_to_bf16_bits(x).astype(np.uint32) << 16).view(np.float32).reshape(x.shape)).astype(np.float64) @ w[finite].astype(np.float64).T
    assert np.all(np.abs(got[:, finite] - want) <= K * 2.0 ** -24 * np.abs(w[finite]).astype(np.float64).sum(1))  # (fp32 sums in any order; |x| <= 1)
    ctx.L.ps_hip_dense_free(ctx.h, h)
    dx.free(); do.free()


# the scratch that a product of many rows takes belongs to the context and stays: it has a bound, and the product goes through it piece by piece
@pytest.mark.parametrize("dtype,T,N,K", [("bfloat16", 40000, 24, 2048), ("float32", 20001, 24, 2048), ("float32 lines", 20001, 24, 2048), ("bfloat16", 1100000, 8, 16)])
def test_dense_matmul_scratch_is_bounded(free_bytes, dtype, T, N, K):
    import ctypes as C
    own = hip.Ctx(0)
    rng = np.random.default_rng(3)
    bits = f32_to_bf16_bits(rng.standard_normal((N, K), dtype=np.float32))
    x = rng.standard_normal((64, K), dtype=np.float32)[np.arange(T) % 61]  # (61 different rows)
    h = C.c_void_p()
    own.check(own.L.ps_hip_dense_upload(own.h, bits.ctypes.data_as(C.c_void_p), N, K, FORMS[dtype], C.byref(h)))
    dx, do = own.to_device(x), own.to_device(np.zeros((T, N), np.float32))
    before = free_bytes()
    own.check(own.L.ps_hip_dense_matmul(own.h, h, dx.ptr, T, do.ptr, 1.0))
    got = do.numpy()
    assert before - free_bytes() <= 100 << 20  # 64 MiB of rows, 32 MiB of parts of split products
    w = (bits.astype(np.uint32) << 16).view(np.float32).reshape(N, K).astype(np.float64)
    a = ((f32_to_bf16_bits(x[:61]).astype(np.uint32) << 16).view(np.float32).reshape(61, K) if dtype == "bfloat16" else x[:61]).astype(np.float64)
    bound = K * 2.0 ** -24 * (np.abs(a) @ np.abs(w).T)
    assert np.all(np.abs(got - (a @ w.T)[np.arange(T) % 61]) <= bound[np.arange(T) % 61])
    own.L.ps_hip_dense_free(own.h, h)
    dx.free(); do.free()
    own.close()


# a latent layer's window is expanded with the same kernel, however few tokens the model takes at a time: the same portions give the same bits
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_model_of_few_tokens_takes_the_same_kernels(made, dtype):
    cfg = synth.seq_config(64, 40, [L("latent_attention", None, heads=4, dim=32, vdim=48, q_rank=20, kv_rank=1088, mask={"size": 70}, scale=0.2, rot={"base": 100.0, "dims": 8}, rot_dim=16)], taps=2)
    toks = tokens_for(cfg, 120)
    few, c, t = made("few", dtype, max_batch=8, cfg=cfg)
    many, _, _ = made("few", dtype, max_batch=32, cfg=cfg, tensors=t)
    for sizes in ((8,), (2, 5, 8)):
        got = run_portions(few, toks, sizes)
        assert np.array_equal(got, run_portions(many, toks, sizes)), sizes
        assert err(got, seq_oracle.run(c, t, toks)) < TOL[dtype]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["wkv", "delta", "latent", "ff", "mixed", "aligned", "wide_heads"])
def test_whole_prompt_against_the_plain_statement(made, name, dtype):
    m, cfg, t = made(name, dtype, max_batch=64)
    toks = tokens_for(cfg, 41)
    want = seq_oracle.run(cfg, t, toks)
    s = m.acquire()
    got = m.forward(s, toks, np.arange(len(toks)))
    m.release(s)
    assert err(got, want) < TOL[dtype]


@pytest.mark.parametrize("name", ["mixed", "aligned", "wide_heads"])
def test_residual_stream_after_every_layer(made, name):
    m, cfg, t = made(name, "float32", max_batch=64)
    toks = tokens_for(cfg, 20, seed=5)
    per = []
    seq_oracle.run(cfg, t, toks, per_layer=per)
    m.capture_layers(True)
    s = m.acquire()
    m.forward(s, toks)
    got = m.layers(len(toks))
    m.release(s)
    m.capture_layers(False)
    for i, want in enumerate(per):
        assert np.abs(got[i] - want).max() < 2e-4 * np.abs(want).max(), i


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["mixed", "aligned", "wide_heads"])
def test_token_by_token_and_portions_give_the_whole_prompts_logits(made, name, dtype):
    m, cfg, t = made(name, dtype, max_batch=16)  # 16: a 50-token portion is also cut inside the library
    toks = tokens_for(cfg, 75, seed=2)
    want = seq_oracle.run(cfg, t, toks)
    for sizes in ([1], [2], [3, 1, 7, 2], [50, 2, 23], [16, 17, 15]):
        assert err(run_portions(m, toks, sizes), want) < TOL[dtype], sizes


def test_first_tokens_of_a_sequence(made):
    """sequences shorter than any convolution's taps, alone and as the start of a longer one"""
    m, cfg, t = made("aligned", "float32")
    for n in (1, 2, 3):
        toks = tokens_for(cfg, n, seed=10 + n)
        assert err(run_portions(m, toks, [n]), seq_oracle.run(cfg, t, toks)) < TOL["float32"]
        assert err(run_portions(m, toks, [1]), seq_oracle.run(cfg, t, toks)) < TOL["float32"]


def test_results_of_a_call_of_several_portions(made):
    """wanted rows that repeat, up to max_batch of them; rows of a portion too many for a half of the pinned memory between portions whose rows fit, portions without any"""
    cfg = synth.seq_config(40, 40000, [L("wkv", 24, heads=1, dim=8)], taps=2)
    m, cfg, t = made("40000", "float32", max_batch=16, cfg=cfg)
    toks = tokens_for(cfg, 75, seed=3)
    rows = seq_oracle.run(cfg, t, toks)
    s = m.acquire()
    for want in (np.array([0, 0, 3] + list(range(16, 32)) + [48, 63, 63] + [70]), np.full(16, 5), np.array([2] * 16 + [74] * 11)):
        for argmax in (False, True):
            m.release(s)
            s = m.acquire()
            got = m.forward(s, toks, want=want, argmax=argmax)
            assert m.position(s) == 75
            if argmax:
                assert np.array_equal(got, ids)
            else:
                assert err(got, rows[want]) < TOL["float32"]
                ids = got.argmax(-1)
    m.release(s)
    s = m.acquire()
    with pytest.raises(hip.PSHipError, match="wanted rows"):
        m.forward(s, toks, want=np.full(17, 40))
    assert m.position(s) == 0
    m.release(s)


# inputs longer than max_batch, whose launch sequences take up to four times as many tokens (seq_rows): every row wanted, more than the head takes at a time; a last one of a single token; a width of four
# times max_batch that the context cuts; rows of a second group that repeat
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("max_batch,n,max_context", [(64, 300, 1024), (64, 257, 1024), (150, 420, 500), (63, 200, 1024)])
def test_a_long_input_in_launch_sequences_wider_than_max_batch(ctx, tmp_path, dtype, max_batch, n, max_context):
    cfg = CONFIGS["mixed"]
    t = synth.write_seq_model_dir(str(tmp_path), cfg, 0, None)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype=dtype, max_batch=max_batch, n_slots=1, max_context=max_context)
    assert m.launch_rows == {64: 256, 150: 500, 63: 63}[max_batch]
    toks = tokens_for(cfg, n, seed=6)
    # (bfloat16: against calls of max_batch tokens.  Rounding alone moves row 151 by 0.1175, in portions of any size and token by token; another cut may round it the other way: a tenth of that)
    rows, tol = (seq_oracle.run(cfg, t, toks), TOL[dtype]) if dtype == "float32" else (run_portions(m, toks, (max_batch,)), 0.012)
    for want in (np.arange(n), np.array([0] * max_batch + [max_batch] * max_batch + [n - 1] * 3)):
        s = m.acquire()
        assert err(m.forward(s, toks, want), rows[want]) < tol
        assert m.position(s) == n
        m.release(s)
    assert err(run_portions(m, toks, (n - 1, 1)), rows) < tol
    m.close()


# a head of more rows than the embedding has: a generated id beyond them embeds as zeros (k_dense.hip dense_next_kernel), the ones in front of it as their rows; eager and captured
@pytest.mark.parametrize("mode", [0, 1])
def test_a_generated_id_without_a_row_of_the_embedding(ctx, tmp_path, mode):
    cfg = synth.seq_config(48, 300, [L("wkv", 40, heads=2, dim=24)], taps=2)
    t = synth.seq_tensors(cfg, 3)
    t["embed"], t["head"] = t["embed"][:20], t["head"].copy()
    t["head"][:280] = 0  # (so that every generated id is one of the last twenty)
    synth.write_seq_model_dir(str(tmp_path), cfg, 3, t)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=8, n_slots=2)
    t = {n: (f32_to_bf16_bits(a).astype(np.uint32) << 16).view(np.float32).reshape(np.shape(a)) for n, a in t.items()}
    t["embed"] = np.concatenate([t["embed"], np.zeros((280, 48), np.float32)])
    m.set_mode(mode)
    s = m.acquire()
    ids = m.decode_greedy(s, 7, 4)
    want = seq_oracle.run(cfg, t, np.array([7, *ids[:3]]))
    assert ids.min() >= 280 and np.array_equal(ids, want.argmax(-1))
    with pytest.raises(hip.PSHipError):
        m.forward(s, ids[-1:], [0])
    m.close()


def test_interleaved_requests_and_reused_slots(made):
    m, cfg, t = made("mixed", "float32", max_batch=16)
    seqs = [tokens_for(cfg, n, seed=20 + n) for n in (37, 9, 58)]
    want = [seq_oracle.run(cfg, t, s) for s in seqs]
    sched = seqmodel.RequestScheduler(m)
    got, at = [[] for _ in seqs], [0, 0, 0]
    steps = [5, 2, 11, 1, 3]
    i = 0
    while any(a < len(s) for a, s in zip(at, seqs)):
        r = i % 3
        if at[r] < len(seqs[r]):
            n = min(steps[i % len(steps)], len(seqs[r]) - at[r])
            got[r].append(sched.feed("req%d" % r, seqs[r][at[r]:at[r] + n], np.arange(n)))
            at[r] += n
            if at[r] == len(seqs[r]):
                sched.finish("req%d" % r)
        i += 1
    for g, w in zip(got, want):
        assert err(np.concatenate(g), w) < TOL["float32"]
    # every slot has been used: a new request gets a used one and must start from nothing
    for r in range(4):
        assert err(sched.feed("again", seqs[2], np.arange(len(seqs[2]))), want[2]) < TOL["float32"]
        sched.finish("again")
    with pytest.raises(hip.PSHipError):
        [m.acquire() for _ in range(4)]
    for s in range(3):
        m.release(s)


def peaked_latent_model(window, seed=0, second_layer=True, aligned=False):
    """A latent-attention model whose scores are made by hand: every token's embedding is a constant half (ones) and a token-specific half of
    +-1 (so the norm in front of the mixer changes nothing); queries and the shared rotated key part read the constant half only, so the rotated
    part of the score depends on the DISTANCE alone, 8 (cos(d) + cos(2 pi d / (window - 1))) for window - 1 = 44 k: largest for the token
    itself and for the key at the far edge of the window (44 k is a whole number of turns of the first pair, up to 0.02 rad).  Values read the
    token-specific half.  A key lost or gained at the edge therefore moves the output by a large fraction of itself."""
    rng = np.random.default_rng(seed)
    W, half, V, H, d, dv, qr, kr, dr = 16, 8, 32, 2, 4, 6, 4, 6, 4
    if aligned:  # sizes the matrix-core attention kernels take (the prompt's and the absorbed single-token form); 4 of 16 rotated numbers turn
        d, dv, kr, dr = 16, 8, 16, 16
    f1 = 2 * np.pi / (window - 1)
    mixer = dict(heads=H, dim=d, vdim=dv, q_rank=qr, kv_rank=kr, rot_dim=dr, rot={"base": float(1.0 / f1 ** 2), "dims": 4}, mask={"size": int(window)}, scale=2.0)
    layers = [synth.seq_layer("latent_attention", None, **mixer)] + ([synth.seq_layer("wkv", 24, heads=2, dim=8)] if second_layer else [])
    cfg = synth.seq_config(W, V, layers, taps=1)
    t = synth.seq_tensors(cfg, seed)
    t["embed"] = np.concatenate([np.ones((V, half)), rng.choice([-1.0, 1.0], (V, W - half))], 1).astype(np.float32)
    for n in ("l0.norm1", "l0.canon1"):
        t[n] = np.zeros_like(t[n])
    dq = np.zeros((qr, W), np.float32)
    dq[:, :half] = rng.standard_normal((qr, half)) * 0.5
    t["l0.mix.dq"], t["l0.mix.dq.norm"] = dq, np.ones(qr, np.float32)
    c0 = dq[:, :half].sum(1).astype(np.float64)
    c0 = c0 / np.sqrt(np.mean(c0 * c0) + cfg["norm"]["eps"])       # the query latent of every token
    uq = rng.standard_normal((H, d + dr, qr)) * 0.1
    uq[:, d:, :] = np.outer([2.0, 2.0] + [0.0] * (dr - 2), c0 / (c0 @ c0))   # rotated query part (2, 2, 0, ...) before the rotation
    t["l0.mix.uq"] = uq.reshape(H * (d + dr), qr).astype(np.float32)
    dkv = np.zeros((kr + dr, W), np.float32)
    dkv[:kr, half:] = rng.standard_normal((kr, W - half)) * 0.5     # the latent reads the token-specific half
    dkv[kr:kr + 2, :half] = 2.0 / half                              # shared key part (2, 2, 0, 0) before the rotation
    t["l0.mix.dkv"] = dkv
    t = {k: (f32_to_bf16_bits(np.asarray(v, np.float32)).astype(np.uint32) << 16).view(np.float32).reshape(np.shape(v)) for k, v in t.items()}
    return cfg, t


def _rows(got, want, lo):
    return [err(got[i:i + 1], want[i:i + 1]) for i in range(lo, len(want))]


@pytest.mark.parametrize("aligned", [False, True])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_window_edges_in_prompts_and_in_decoding(made, dtype, aligned):
    """The plain statement with a window one shorter loses the edge key and is far off at every later position, one longer gains a key and is
    clearly off; the library agrees with the right one whether the edge passes over prompt tokens, portions' borders or decoded tokens, also
    when the ring of latents (window - 1 + 8 rows here) has wrapped."""
    window = 45
    cfg, t = peaked_latent_model(window, aligned=aligned)
    m, _, _ = made("peaked45%d" % aligned, dtype, max_batch=8, cfg=cfg, tensors=t)
    toks = tokens_for(cfg, 120, seed=3)
    want = seq_oracle.run(cfg, t, toks)
    assert np.median(_rows(seq_oracle.run(cfg, t, toks, window_override={0: window - 1}), want, window - 1)) > 0.3
    assert np.median(_rows(seq_oracle.run(cfg, t, toks, window_override={0: window + 1}), want, window)) > 5e-3
    for sizes in ([120], [1], [8], [5, 2, 12, 1], [43, 1, 1, 1, 1, 1], [44, 2, 1], [46, 1]):
        got = run_portions(m, toks, sizes)
        assert max(_rows(got, want, 0)) < (1e-3 if dtype == "float32" else TOL[dtype]), sizes


@pytest.mark.parametrize("aligned", [False, True])
def test_far_key_among_hundreds_and_a_ring_that_wraps(made, aligned):
    """window 309: the key 308 tokens back carries a large share of the weight.  A 330-token prompt in portions of 64, then 170 single tokens:
    the ring (372 rows) wraps, and the far key is first a prompt token, then a decoded one."""
    window = 309
    cfg, t = peaked_latent_model(window, seed=1, aligned=aligned)
    m, _, _ = made("peaked309%d" % aligned, "float32", max_batch=64, cfg=cfg, tensors=t)
    toks = tokens_for(cfg, 500, seed=4)
    want = seq_oracle.run(cfg, t, toks)
    assert np.median(_rows(seq_oracle.run(cfg, t, toks, window_override={0: window - 1}), want, window - 1)) > 0.1
    s = m.acquire()
    got = [m.forward(s, toks[:330], np.arange(330))] + [m.forward(s, toks[i:i + 1], [0]) for i in range(330, 500)]
    m.release(s)
    assert max(_rows(np.concatenate(got), want, 0)) < 1e-3


def test_long_decoding_keeps_the_recurrent_states(made):
    m, cfg, t = made("mixed", "float32", max_batch=16)
    toks = tokens_for(cfg, 260, seed=6)
    want = seq_oracle.run(cfg, t, toks)
    assert err(run_portions(m, toks, [13, 1, 1, 1, 1, 1, 1, 1]), want) < TOL["float32"]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_greedy_generation_through_the_entry_point(made, dtype):
    """SeqModel.generate (prefill, then the captured single-token step feeding its own arg-max) picks, at every step, a token whose logit in the
    plain statement is the largest up to rounding; eager launches and a host sampler set to top-1 give the same ids."""
    m, cfg, t = made("mixed", dtype, max_batch=16)
    prompt = tokens_for(cfg, 19, seed=7)
    ids = m.generate(prompt, 24)
    assert ids.shape == (24,)
    full = np.concatenate([prompt, ids])
    want = seq_oracle.run(cfg, t, full[:-1])
    spread = want.max() - want.min()
    for i, tok in enumerate(ids):
        row = want[len(prompt) - 1 + i]
        assert row.max() - row[tok] < (1e-4 if dtype == "float32" else 3e-2) * spread, i
    m.set_mode(1)
    assert np.array_equal(m.generate(prompt, 24), ids)
    m.set_mode(0)
    assert np.array_equal(m.generate(prompt, 24), ids)  # the captured sequence replayed on a slot that was used before
    sm = host.Sampler(host.SamplerCfg.make(cfg["vocab"], seed=1, temperature=1.0, top_p=1.0, top_k=1))
    assert np.array_equal(m.generate(prompt, 24, sampler=sm.sample), ids)
    sm.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_matrix_core_forms_agree_with_the_plain_kernels(made, dtype):
    """mode bit 1 keeps the per-key attention, the expanded single-token step and the 64 x 64 mat-mul: the wide mat-mul, the matrix-core
    attention of a portion and the absorbed single-token attention must give the same logits (fp32: up to the order of sums)"""
    m, cfg, t = made("aligned", dtype, max_batch=64)
    toks = tokens_for(cfg, 150, seed=9)
    fast = [run_portions(m, toks, sizes) for sizes in ([64], [1], [40, 1, 1, 1, 9])]
    m.set_mode(2)
    plain = [run_portions(m, toks, sizes) for sizes in ([64], [1], [40, 1, 1, 1, 9])]
    m.set_mode(0)
    want = seq_oracle.run(cfg, t, toks)
    for a, b in zip(fast, plain):
        assert err(a, b) < (1e-4 if dtype == "float32" else TOL[dtype])
        assert err(a, want) < TOL[dtype]


def test_host_facade_loads_and_generates_the_same(made, tmp_path):
    """load_seq_model of the C++ facade (its own safetensors reader and configuration mapping) over the same files: same ids, same logits"""
    m, cfg, t = made("mixed", "float32", max_batch=16)
    synth.write_seq_model_dir(str(tmp_path), cfg, 0, t)
    assert host.lib().psh_is_seq_model_dir(str(tmp_path).encode()) == 1
    hm = host.HostSeqModel(str(tmp_path), dtype="float32", max_batch=16, n_slots=2)
    prompt = tokens_for(cfg, 19, seed=7)
    ids = m.generate(prompt, 12)
    assert np.array_equal(hm.generate(prompt, 12), ids)
    assert np.array_equal(hm.generate(prompt, 12, host.SamplerCfg.make(cfg["vocab"], seed=3, temperature=1.0, top_p=1.0, top_k=1)), ids)
    s, s2 = hm.acquire(), m.acquire()
    a, b = hm.forward(s, prompt, [0, 5, 18]), m.forward(s2, prompt, [0, 5, 18])
    hm.release(s)
    m.release(s2)
    assert np.array_equal(a, b)
    with pytest.raises(host.HostError):
        host.HostModel(str(tmp_path))  # the quantized path's loader says what this folder is instead of looking for model.json
    hm.close()


def test_refusals(ctx, tmp_path):
    cfg = dict(CONFIGS["wkv"])
    synth.write_seq_model_dir(str(tmp_path), cfg, 0)
    m = seqmodel.load_model(ctx, str(tmp_path), dtype="float32", max_batch=4, n_slots=1)
    s = m.acquire()
    with pytest.raises(hip.PSHipError):
        m.forward(s, [cfg["vocab"]])
    with pytest.raises(hip.PSHipError):
        m.forward(s + 1, [0])
    m.release(s)
    with pytest.raises(hip.PSHipError):
        m.release(s)
    m.close()
