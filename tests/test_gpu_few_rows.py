"""GPU parity of the encoder on batches of few rows, whose Wo and MLP
products run cut by output channel (split_rows.hip), against the CPU
oracle, bit for bit."""
import concurrent.futures as cf

import numpy as np
import pytest

from helpers import base_cfg, bekko_cfg, f32_bits_equal, mismatch_report, small_cfg
from indecis_amd.modernbert import Model, Weights
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SHAPES = {"small": small_cfg, "base": base_cfg, "bekko": bekko_cfg}


def seqs_of(rng, vocab, *lens):
    return [rng.integers(0, vocab, size=n, dtype=np.int32) for n in lens]


# shape, lane width, rows past the dequantisation bound planted in a matrix
@pytest.mark.parametrize("shape,lanes,plant", [
    ("base", 8, None), ("base", 16, "wo"), ("base", 0, "womlp"), ("bekko", 8, "wi"), ("bekko", 4, None),
    ("bekko", 16, None), ("bekko", 0, None),
    ("small", 8, "wo"), ("small", 16, None), ("small", 4, "womlp"), ("small", 0, "wi")])
def test_few_rows_exact(shape, lanes, plant):
    """Row counts around the 32-row blocks (and the 8 rows of a LayerNorm
    workgroup), one sequence or several, a sequence over 512 keys (QKV input
    row-major), the LayerNorm in the Wi kernel and before it (up to 192 rows,
    shape small 512), the two arrangements of the residual kernel (from 481 rows
    on) and the two sides of the rules that pick these kernels and the
    32-row MLP kernel; option few_rows 0 picks the whole-row kernels, and gives
    the same bits."""
    cfg = SHAPES[shape](layers=2)
    w = Weights.random(cfg, seed=97)
    if plant:
        {"wi": w.wi_q, "wo": w.wo_q, "womlp": w.womlp_q}[plant][0, 3, :] = 127
    gpu, ora = Model(w, lanes=lanes), orc.OracleModel(w, lanes=lanes)
    rng = np.random.default_rng(97)
    batches = [seqs_of(rng, cfg.vocab, *lens)
               for lens in ((1,), (7, 1), (31,), (9, 0, 23), (33,), (192,), (193,), (64, 1, 192), (480,), (481,), (512,), (513,), (600, 9))]
    gpu.set_option("parts", 1)
    want = [ora.encode_tokens(b)[0] for b in batches]
    for b, e in zip(batches, want):
        got = gpu.encode_tokens(b)
        assert f32_bits_equal(got, e), ([len(s) for s in b], mismatch_report(got, e))
    most = {"small": 2048, "base": 3072, "bekko": 4096}[shape]
    edges = [seqs_of(rng, cfg.vocab, *[64] * (n // 64), n % 64) for n in (most, most + 1, 8192, 8193)]
    few = [gpu.encode_tokens(b) for b in batches + edges]
    gpu.set_option("few_rows", 0)
    for b, e in zip(batches + edges, few):
        got = gpu.encode_tokens(b)
        assert f32_bits_equal(got, e), ([len(s) for s in b], mismatch_report(got, e))
    gpu.close()


@pytest.mark.parametrize("shape,lanes,window,plant", [
    ("small", 8, 128, False), ("small", 0, 16, True), ("small", 16, 16, False), ("small", 4, 128, True),
    ("bekko", 8, 16, False), ("bekko", 16, 128, True), ("base", 8, 128, False), ("base", 4, 16, True)])
def test_short_sequences_exact(shape, lanes, window, plant):
    """QKV, Attn8.Prepare and attention in one kernel (short_attn.hip): the
    longest sequence at the edges of its 1, 2 and 4 row blocks, with a local
    window that cuts sequences and one that does not, empty sequences, QKV
    rows past the dequantisation bound, and with the LayerNorm before it in the
    same kernel (at most 32 tokens, 24 rows at a time, one round of the 256
    CUs), against the oracle; and batches one workgroup either side of the rules
    that pick it, by the kernels that ran."""
    cfg = SHAPES[shape](layers=2, local_attention=window)
    w = Weights.random(cfg, seed=101)
    if plant:
        for row in (3, cfg.hidden + 5, 2 * cfg.hidden + 7):
            w.wqkv_q[0, row, :] = 127
    gpu, ora = Model(w, lanes=lanes), orc.OracleModel(w, lanes=lanes)
    rng = np.random.default_rng(101)
    batches = [(1,), (15, 2), (31, 0, 1), (32, 32, 17), (33, 5), (40, 0, 63, 1), (64, 33), (65, 31), (97, 8), (127,),
               (128, 1, 90), (129, 3)]
    one = 256 // cfg.heads
    batches += [(24,), (25, 24, 3), (30,) + (2,) * (one - 1), (30,) + (2,) * one]
    picked = [None] * len(batches)
    # longest sequence, most (or, negative, one less than the fewest) sixteenths of a round
    edges = [(32, 96 if shape == "small" else 80), (64, 32), (65, {"base": -6, "bekko": -4, "small": -2}[shape]), (128, 16)]
    edges += [(33, 16), (64, -28)] if shape == "base" else []
    for n, most in edges:
        seqs = abs(most) * 16 // cfg.heads
        batches += [(n,) + (2,) * (seqs - 1), (n,) + (2,) * seqs]
        picked += [most > 0, most < 0]
    gpu.set_profiling(True)
    for lens, short in zip(batches, picked):
        seqs = seqs_of(rng, cfg.vocab, *lens)
        got, want = gpu.encode_tokens(seqs), ora.encode_tokens(seqs)[0]
        assert f32_bits_equal(got, want), (lens[:4], mismatch_report(got, want))
        ran = set(gpu.profile())
        gpu.set_profiling(True)  # clears the sums
        if short is not None:
            assert ("gemm_qkv" not in ran) == short, (lens[0], len(lens))
    gpu.close()


@pytest.mark.parametrize("shape,tokens,seqs", [
    ("small", 32, 640), ("small", 64, 192), ("bekko", 32, 212), ("bekko", 16, 256), ("base", 128, 42)])
def test_short_sequences_in_parts(shape, tokens, seqs):
    """A batch run as two parts: short_attn.hip up to `seqs` sequences of these
    lengths (its rounds of the 256 CUs a part), with the same bits as the other
    kernels."""
    cfg = SHAPES[shape](layers=2)
    gpu = Model(Weights.random(cfg, seed=102))
    rng = np.random.default_rng(102)
    gpu.set_option("parts", 2)
    for n, short in ((seqs, True), (seqs + 2, False)):
        batch = seqs_of(rng, cfg.vocab, *[tokens] * n)
        gpu.set_profiling(True)
        got = gpu.encode_tokens(batch)
        assert ("gemm_qkv" not in gpu.profile()) == short, n
        gpu.set_profiling(False)
        gpu.set_option("few_rows", 0)
        want = gpu.encode_tokens(batch)
        gpu.set_option("few_rows", 1)
        assert f32_bits_equal(got, want), (n, mismatch_report(got, want))
    gpu.close()


@pytest.mark.parametrize("shape", ["base", "bekko", "small"])
def test_rows_in_parts(shape):
    """A batch run as two parts, which share the CUs: the products cut by output
    channel at hidden 384 up to 5,000 rows in all or in the smaller part (not of
    equal ones) up to 8,192, at 768 in a smaller part of up to 2,304, by the kernels
    that ran; with the same bits as the options' kernels either side of that and of
    the rule of the 32-row MLP kernel."""
    cfg = SHAPES[shape](layers=2)
    gpu = Model(Weights.random(cfg, seed=105))
    rng = np.random.default_rng(105)
    gpu.set_option("parts", 2)
    for rows in (4096, 4500, 5000, 5001, 5120, 8191, 10240, 10241, 16384, 16385):
        batch = seqs_of(rng, cfg.vocab, *[256] * (rows // 256), rows % 256)
        gpu.set_profiling(True)
        got = gpu.encode_seqs(batch)
        ran = set(gpu.profile())
        gpu.set_profiling(False)
        assert ("gemm_womlp" in ran) == (rows in {"bekko": (4096, 4500, 5000, 5001, 8191), "base": (4500,), "small": ()}[shape]), (rows, ran)
        gpu.set_option("few_rows", 0)
        want = gpu.encode_seqs(batch)
        gpu.set_option("few_rows", 1)
        assert f32_bits_equal(got, want), (rows, mismatch_report(got, want))
    gpu.close()


@pytest.mark.parametrize("shape", ["base", "small"])
def test_rows_beside_threads(shape):
    """Threads calling one handle, whose passes share the CUs and so pick other
    kernels than alone (whole rows for passes of some thousand rows), by the
    kernels that ran; with the bits of calls one at a time, and the kernels of a
    call alone afterwards."""
    cfg = SHAPES[shape](layers=2)
    gpu = Model(Weights.random(cfg, seed=106))
    rng = np.random.default_rng(106)
    gpu.set_option("parts", 1)
    batches = [seqs_of(rng, cfg.vocab, *lens) for lens in
               ([256] * 8, [200] * 10, [16, 24] * 12, [64] * 3, [15], [256] * 7 + [255], [33] * 20, [2000])]
    gpu.set_profiling(True)
    want = [gpu.encode_seqs(b) for b in batches]
    assert "mlp_ln" not in gpu.profile()
    gpu.set_profiling(True)
    with cf.ThreadPoolExecutor(len(batches)) as ex:
        for b, e, got in zip(batches, want, ex.map(lambda b: [gpu.encode_seqs(b) for _ in range(12)], batches)):
            assert all(f32_bits_equal(g, e) for g in got), [len(s) for s in b][:4]
    assert "mlp_ln" in gpu.profile()
    gpu.set_profiling(True)
    gpu.encode_seqs(batches[3])
    assert "ln_wi" in gpu.profile()
    gpu.close()


@pytest.mark.parametrize("shape,window", [("small", 128), ("bekko", 30)])
def test_shared_keys_exact(shape, window):
    """Attention with 1, 2 and 4 waves on a query block's keys
    (attention_i8.hip), by the number of query blocks and the longest
    sequence: one sequence around the chunks of 256 keys and past 512 keys,
    and batches either side of 256 and of 512 workgroups, against the oracle
    (the largest against one-sequence calls)."""
    cfg = SHAPES[shape](layers=2, local_attention=window)
    w = Weights.random(cfg, seed=103)
    gpu, ora = Model(w), orc.OracleModel(w)
    rng = np.random.default_rng(103)
    for lens in ((129,), (255, 3), (256, 130), (257,), (512, 2), (513,), (545, 40), (1025, 1)):
        seqs = seqs_of(rng, cfg.vocab, *lens)
        got, want = gpu.encode_tokens(seqs), ora.encode_tokens(seqs)[0]
        assert f32_bits_equal(got, want), (lens, mismatch_report(got, want))
    gpu.set_option("parts", 1)
    for items in (256, 512):
        for blocks in (items // cfg.heads, items // cfg.heads + 1):
            seqs = seqs_of(rng, cfg.vocab, *[150, 129] * (blocks // 4), *[140] * ((blocks % 4) // 2), *[9] * (blocks % 2))
            got = gpu.encode_seqs(seqs)
            want = np.concatenate([gpu.encode_seqs([s]) for s in seqs])
            assert f32_bits_equal(got, want), (blocks, mismatch_report(got, want))
    gpu.close()


@pytest.mark.parametrize("shape,lanes,plant", [("small", 8, False), ("bekko", 16, True), ("base", 8, False)])
def test_shared_qkv_workgroups_exact(shape, lanes, plant):
    """The fused QKV kernel's workgroups shared by sequences of at most 256
    tokens (qkv_groups): random lengths, every padded block count beside every
    other, empty sequences between and at the end, sequences over 256 tokens
    among them, and QKV rows past the dequantisation bound, against the
    oracle."""
    cfg = SHAPES[shape](layers=2)
    w = Weights.random(cfg, seed=107)
    if plant:
        w.wqkv_q[0, cfg.hidden + 5, :] = 127
    gpu, ora = Model(w, lanes=lanes), orc.OracleModel(w, lanes=lanes)
    rng = np.random.default_rng(107)
    # (shared from 512 workgroups on: 3 * heads a sequence; groups of 16 blocks
    # with a sequence over 256 tokens or past 2,048 workgroups)
    batches = [(129, 64, 1, 128, 0, 65, 192, 2, 256, 0), (193, 63, 130, 127, 33, 257, 31, 32, 512, 0, 0),
               tuple(int(n) for n in rng.integers(0, 300, 60 if shape == "small" else 30)) + (0,),
               tuple(int(n) for n in rng.integers(0, 257, 60 if shape == "small" else 20)) + (0, 256)]
    for lens in batches:
        seqs = seqs_of(rng, cfg.vocab, *lens)
        got, want = gpu.encode_tokens(seqs), ora.encode_tokens(seqs)[0]
        assert f32_bits_equal(got, want), (lens, mismatch_report(got, want))
        assert f32_bits_equal(gpu.encode_seqs(seqs), ora.encode_seqs(seqs)), lens
    if shape == "small":
        gpu.set_option("parts", 1)
        seqs = seqs_of(rng, cfg.vocab, *(int(n) for n in rng.integers(129, 257, 200)))
        got, want = gpu.encode_tokens(seqs), ora.encode_tokens(seqs)[0]
        assert f32_bits_equal(got, want), mismatch_report(got, want)
    gpu.close()


@pytest.mark.parametrize("rows", [5888, 5889])
def test_final_norm_four_lanes(rows):
    """The final LayerNorm of 4 lanes at hidden 768 either side of the row count
    at which its kernel changes, against the options' kernels."""
    cfg = base_cfg(layers=1)
    gpu = Model(Weights.random(cfg, seed=111), lanes=4)
    gpu.set_option("parts", 1)
    seqs = seqs_of(np.random.default_rng(111), cfg.vocab, *[128] * (rows // 128), rows % 128)
    got = gpu.encode_tokens(seqs)
    gpu.set_option("few_rows", 0)
    want = gpu.encode_tokens(seqs)
    assert f32_bits_equal(got, want), mismatch_report(got, want)
    gpu.close()


def test_options_set_back():
    """An option read, changed and set back leaves a handle with the kernels of
    few rows that it had, and so does few_rows."""
    cfg = small_cfg(layers=2)
    gpu = Model(Weights.random(cfg, seed=109))
    seqs = seqs_of(np.random.default_rng(109), cfg.vocab, 24)

    def classes():
        gpu.set_profiling(True)
        gpu.encode_seqs(seqs)
        got = set(gpu.profile())
        gpu.set_profiling(False)
        return got

    few = classes()
    assert "ln_wi" in few
    for name, other in (("fuse_mlp", 1), ("gemm_tile", 1), ("few_rows", 0)):
        old = gpu.option(name)
        gpu.set_option(name, other)
        assert "ln_wi" not in classes(), name
        gpu.set_option(name, old)
        assert classes() == few, name
    gpu.close()
