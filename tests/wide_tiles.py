"""Sizes at which the wide mat-mul (k_dense.hip dn_ring_plan) takes each of its tiles.  test_host_calls.py counts the launches of these products by the kernel's name, test_gpu_seq.py runs them: a rule that moves one
of them to other tiles fails the first, so that the second goes on reaching every form."""

# {(matrix format, tile rows, tile columns): [(tokens, outputs, K, parts of K or one)]}.  Tiles of 256 columns: one block of K (64 numbers), two, three, five and nine; a row and four columns more than a tile, a column more and
# two or three (no fours), a whole one.  Parts: even and uneven shares.
PRODUCTS = {
    ("bfloat16", 256, 256): [(577, 16388, 64, 1), (600, 16640, 192, 1), (641, 16385, 320, 1), (577, 18435, 576, 1)],
    ("bfloat16", 192, 256): [(385, 16388, 64, 1), (449, 16640, 192, 1), (641, 14338, 192, 1), (385, 16385, 576, 1)],
    ("bfloat16", 128, 256): [(385, 14340, 64, 1), (193, 16388, 192, 1), (449, 12289, 320, 1), (257, 16640, 576, 1), (193, 16385, 576, 1)],
    ("bfloat16", 192, 128): [(257, 12292, 1088, 1), (257, 12290, 1152, 1), (129, 6148, 3136, 5), (150, 6149, 4160, 5)],
    ("bfloat16", 128, 128): [(193, 8196, 576, 1), (193, 2052, 4096, 6), (200, 2053, 4160, 6)],
    ("bfloat16", 64, 128): [(193, 4100, 1088, 1), (193, 2052, 3136, 3), (300, 2048, 4096, 3), (385, 1029, 4096, 4)],
    ("bfloat16", 64, 64): [(65, 129, 320, 1), (300, 512, 64, 1), (129, 513, 1600, 5)],
    ("float32 lines", 256, 256): [(641, 16388, 128, 1), (641, 16388, 192, 1), (641, 16386, 320, 1), (641, 16385, 576, 1)],
    ("float32 lines", 192, 256): [(385, 16388, 64, 1), (385, 16392, 128, 1), (641, 16384, 320, 1), (449, 16385, 1088, 1)],
    ("float32 lines", 192, 128): [(513, 7172, 64, 1), (513, 7173, 576, 1), (513, 3588, 1088, 2), (129, 3588, 2112, 7), (150, 4101, 2112, 7)],
    ("float32 lines", 128, 128): [(193, 8196, 576, 1), (65, 8196, 1088, 3), (65, 6149, 2112, 5)],
    # few tokens: 64 rows in parts, where one round of whole 64 x 64 tiles takes a tenth longer
    ("float32 lines", 64, 128): [(2, 4096, 4096, 8), (8, 8192, 2048, 4)],
}

# An epilogue behind each height of the tiles of 256 columns, and behind 192 x 128 whole and in parts: {(which, format): [(size, tokens, width, rows, columns, in parts)]}.  size: feed-forward numbers, of mixes heads
EPILOGUES = {
    ("xielu", "bfloat16"): [(16384, 400, 576, 128, 256, 0), (16384, 600, 576, 192, 256, 0), (16384, 1000, 192, 256, 256, 0), (8192, 600, 192, 192, 128, 0)],
    ("pairs", "bfloat16"): [(8192, 400, 576, 128, 256, 0), (8192, 600, 576, 192, 256, 0), (8192, 1000, 192, 256, 256, 0)],
    ("experts", "bfloat16"): [(6144, 400, 192, 128, 256, 0), (6144, 600, 192, 192, 256, 0), (6144, 1000, 192, 256, 256, 0)],
    ("mixes", "bfloat16"): [(24, 400, 192, 128, 256, 0), (32, 600, 192, 192, 256, 0), (24, 1000, 192, 256, 256, 0)],
    ("experts", "float32"): [(6144, 600, 192, 192, 256, 0), (12288, 400, 192, 256, 256, 0)],
    ("mixes", "float32"): [(32, 600, 192, 192, 256, 0), (32, 1000, 192, 256, 256, 0)],
    ("pairs", "float32"): [(8192, 600, 192, 192, 128, 0), (2048, 130, 2112, 192, 128, 1)],
    ("xielu", "float32"): [(16384, 600, 192, 192, 128, 0), (4096, 130, 2112, 192, 128, 1)],
}


def layers(synth, which, size, width, vocab=30):
    """the configuration of one layer whose product it is"""
    if which == "experts":
        return synth.pupidra_config(width, vocab, [synth.pupidra_layer("attention", synth.pupidra_attention(2, 1, 16, 16, 0.3, 9, 2), moe=(5, 2, size, 1.7), shared=8)])
    if which == "mixes":
        return synth.seq_config(width, vocab, [synth.seq_layer("wkv", None, heads=size, dim=128)], taps=2)
    if which == "pairs":
        return synth.pokatar_config(width, vocab, [synth.pokatar_layer("attention", synth.pokatar_attention(2, 1, 16, 16, 0.3), size)])
    return synth.seq_config(width, vocab, [synth.seq_layer("delta", size, heads=2, kv_heads=1, dim=16, vdim=16, conv=2)], taps=2)


def kernel(fmt, rows, columns, odd):
    """what the launch's mangled name holds"""
    lines = 1 if fmt == "bfloat16" else 3
    return f"dense_mm_big_kernelILb{odd}ELi{lines}ELi{rows // 64}E" if columns == 256 else f"dense_mm_ring_kernelItLi{rows}ELi{columns}ELb{odd}ELi{lines}E"
