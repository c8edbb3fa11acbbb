"""The C-ABI library on the CPU: it loads, exports every entry point
include/ts5hip.h declares, reports layouts and errors without a GPU, and its
host-side sampler draws exactly as ts5's Engine::sample (engine/src/engine.cpp:16-46).
No GPU compute runs here."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import make_golden
import oracle
from tokenstation5_amd import synth, ts5hip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
G = os.path.join(ROOT, "tests", "golden")


def test_library_exports_every_declared_symbol():
    L = ts5hip.lib()
    syms = ts5hip.header_symbols()
    assert len(syms) >= 40
    missing = [s for s in syms if not hasattr(L, s)]
    assert not missing, missing
    # Every declared function has a ctypes signature in the binding, and vice versa.
    assert set(syms) == set(ts5hip._SIGS)


def test_header_compiles_as_c_and_cxx():
    for cc, flag in (("gcc", "-xc"), ("g++", "-xc++")):
        r = subprocess.run([cc, flag, "-std=c99" if cc == "gcc" else "-std=c++17", "-fsyntax-only", "-Wall",
                            "-Werror", "-I", os.path.join(ROOT, "include"), "-"],
                           input='#include "ts5hip.h"\nint main(void){return 0;}\n', text=True, capture_output=True)
        assert r.returncode == 0, r.stderr


def test_weight_layout_sizes():
    L = ts5hip.lib()
    # Q4_K keeps GGUF's 144 B per 256 values.
    assert L.ts5hip_weight_bytes(ts5hip.Q4_K, 4096, 4096) == 4096 * 16 * 144
    # Split layouts: bodies + f16 scales, each padded to 256 B.
    nb = 128256 * 16
    assert L.ts5hip_weight_bytes(ts5hip.Q6_K, 4096, 128256) == -(-nb * 208 // 256) * 256 + -(-nb * 2 // 256) * 256
    assert L.ts5hip_weight_bytes(ts5hip.Q8_0, 896, 896) == -(-896 * 28 * 32 // 256) * 256 + -(-896 * 28 * 2 // 256) * 256
    assert L.ts5hip_weight_bytes(ts5hip.Q4_K, 100, 4) == -1   # not whole blocks
    # Q4_0, Q4_1, Q5_0, Q5_1, Q5_K: an int8 quant a value and an fp32 (scale, min) pair per 32 values.
    assert L.ts5hip_weight_bytes(13, 256, 4) == 32 * 32 + 32 * 8
    assert L.ts5hip_weight_bytes(2, 32, 9) == 512 + 256
    assert L.ts5hip_weight_bytes(30, 256, 4) == -1           # BF16: not a GPU type of the reference
    # The reference's GPU matrix types (engine/src/vk_backend.cpp:156-170), and not BF16.
    assert [L.ts5hip_supports_type(t) for t in (0, 1, 2, 3, 6, 7, 8, 12, 13, 14, 30)] == [1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0]
    assert L.ts5hip_act_bytes(4096) > 2 * 4096 and L.ts5hip_act_bytes(100) == -1


def test_init_reports_errors_without_gpu():
    if os.path.exists("/dev/kfd"):
        pytest.skip("a GPU is present")
    with pytest.raises(ts5hip.Ts5HipError) as e:
        ts5hip.Context(0)
    assert e.value.code == ts5hip.ERR_HIP


def test_sampler_draw_matches_reference():
    """ts5hip_sampler_draw over the GPU top-k candidate set reproduces the
    reference engine's ids (golden vectors from ts5's own Engine::generate)."""
    s = np.load(os.path.join(G, "sampler.npz"))
    table = make_golden.sampler_table(int(s["table_seed"]), int(s["rows"]), int(s["n_vocab"]))
    for i, (T, p, k) in enumerate(make_golden.SAMPLER_CASES):
        if not (T > 0 and 0 < k <= 64):
            continue
        smp = ts5hip.Sampler(42 + i)
        got = []
        for r in range(table.shape[0]):
            ids = np.argsort(-table[r], kind="stable")[:k].astype(np.int32)
            got.append(smp.draw(ids, table[r][ids], T, p))
        assert got == list(s[f"ids{i}"]), i


def test_rope_table_matches_oracle_angles():
    """The host RoPE table is computed as the CPU path computes its angles;
    checked through the oracle's rope_cs on the CPU (same libm)."""
    import ctypes as C
    L = ts5hip.lib()
    # ts5hip_rope_table needs a context; the angles themselves are pinned via
    # the oracle here and on the GPU by test_gpu_ops.test_rope_kv_append.
    c, s = oracle.rope_cs(128, 4095, 500000.0)
    assert np.isclose(c[0], np.cos(4095.0), atol=1e-3) and np.isclose(s[0], np.sin(4095.0), atol=1e-3)
    assert L.ts5hip_rope_table(None, 128, 16, 500000.0, 1.0, None, None) == ts5hip.ERR_ARG
    del C


def test_synth_layouts_are_whole_blocks():
    for hp in (synth.LLAMA_8B, synth.DRAFT_0P5B, synth.TARGET_14B):
        wb = synth.weight_bytes(hp)
        assert wb["layer"] > 0 and wb["head"] > 0
    # cfg2's per-token weight bytes (algorithmic): 32 Q4_K layers of 4096-wide
    # rows (14336 for down) and the Q6_K head over a 128256-token vocabulary.
    wb = synth.weight_bytes(synth.LLAMA_8B)
    assert wb["layers"] == 3925868544 and wb["head"] == 430940160


def test_prompt_matmul_splits_fit_every_xcd():
    """The prompt matmul's splits of K (wide_splits) run in one round: a unit (row tile, split) and its token
    tiles go to one of the 8 XCDs, units in turn, and an XCD holds 32 of a tile's 8-wave workgroups at a time (64 of the
    4-wave ones that up to 48 tokens take). No split is empty, and one split is always allowed."""
    wide_splits = ts5hip.lib()._ZN6ts5hip11wide_splitsEliiii
    wide_splits.argtypes, wide_splits.restype = [ctypes.c_int64] + [ctypes.c_int] * 4, ctypes.c_int
    many = 0
    for glu in (0, 1):
        for nb in (1, 2, 3, 7, 10, 12, 16, 20, 32, 54, 56):
            for rows in list(range(128, 8192, 384)) + [896, 3072, 7168, 14336, 33000]:
                for M in (17, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 192, 256, 257, 300, 384, 385, 512, 640, 1024):
                    ntt = -(-M // 128)
                    groups = -(-M // ntt)
                    tt = next(t for t in (2, 3, 4, 6, 8) if 16 * t >= groups)
                    ntt = -(-M // (16 * tt))
                    tile = (256 if tt > 3 else 128) // (2 if glu else 1)
                    ks = wide_splits(rows, M, nb, 256, 2 if glu else 1)
                    assert 1 <= ks <= max(1, nb // 2) and ks <= 16, (glu, nb, rows, M, ks)
                    assert (ks - 1) * -(-nb // ks) < nb, (glu, nb, rows, M, ks)
                    units = -(-rows // tile) * ks
                    many += ks > 1
                    assert ks == 1 or -(-units // 8) * ntt <= (32 if tt > 3 else 64), (glu, nb, rows, M, ks)
    assert many > 1000


def test_prompt_attention_partials_bound():
    """attn_prefill_partial_bytes bounds every launch of up to nq queries and max_keys keys: query blocks of
    128 / G queries times the KV heads are a split's workgroups, a launch starts from 512 / workgroups splits of
    at least 256 keys, 16 at most, and takes fewer, longer ones where that saves a round. And it is no more than twice
    what some launch needs."""
    bound = ts5hip.lib()._ZN6ts5hip26attn_prefill_partial_bytesEiiiil
    bound.argtypes, bound.restype = [ctypes.c_int] * 4 + [ctypes.c_int64], ctypes.c_size_t

    def splits(keys, wg):
        want = max(256, -(-keys // max(1, min(16, -(-512 // wg)))))
        first = -(-want // 64) * 64
        best = None
        for per in range(first, 2 * first + 1, 64):
            n = -(-keys // per)
            rounds = per + (0 if wg * n <= 512 else keys - (n - 1) * per if wg * (n - 1) <= 512 else per)
            if best is None or rounds < best[0]:
                best = rounds, n
        return best[1]

    for H, HKV, HD in ((32, 8, 128), (64, 8, 128), (40, 8, 128), (14, 2, 64), (8, 8, 128), (4, 1, 128)):
        for keys in (256, 257, 600, 2048, 4096, 32768):
            need = 0
            for nq in sorted({*range(1, 513, 29), *range(32, 513, 32), *range(25, 513, 25), 512}):
                n = splits(keys, -(-nq // (128 // (H // HKV))) * HKV)
                need = max(need, nq * n * H * (HD + 4) * 4 if n > 1 else 0)
                assert need <= bound(nq, H, HKV, HD, keys), (H, HKV, nq, keys)
            assert bound(512, H, HKV, HD, keys) <= 2 * need, (H, HKV, keys)


def test_fixed_memory_follows_the_buffers(tmp_path):
    """The bytes beside the KV cache that a context is fitted into: the weights, the 512-token buffers with the
    scratch of their matmuls and attention (64 query heads here), 256 logits rows with their picks, 64 MiB."""
    import gguf_writer
    hp = dict(synth.TINY_LLAMA, n_vocab=151936, n_layer=1, n_head=64, n_head_kv=8, head_dim=128)
    tensors = {name: (t, ne0, ne1, np.zeros(synth.row_bytes(t, ne0) * ne1 if t else 4 * ne0 * ne1, np.uint8))
               for name, t, ne0, ne1 in synth.tensor_specs(dict(hp, head_type=None))}
    path = str(tmp_path / "m.gguf")
    gguf_writer.write(path, gguf_writer.model_kv(hp, vocab_pieces=False), tensors)
    fixed = ts5hip.gguf_hparams(path)[2]
    weights = sum(ts5hip.lib().ts5hip_weight_bytes(t, ne0, ne1) if t else 4 * ne0 for t, ne0, ne1, _ in tensors.values())
    E, F, AH, QR, V = 512, 1536, 64 * 128, 80 * 128, 151936
    gemm = ts5hip.lib()._ZN6ts5hip18gemm_scratch_bytesElii
    gemm.argtypes, gemm.restype = [ctypes.c_int64, ctypes.c_int, ctypes.c_int], ctypes.c_size_t
    part = ts5hip.lib()._ZN6ts5hip26attn_prefill_partial_bytesEiiiil
    part.argtypes, part.restype = [ctypes.c_int] * 4 + [ctypes.c_int64], ctypes.c_size_t
    buffers = 4 * 512 * (2 * E + QR + 2 * AH + F) + 512 * 4 * AH
    buffers += max(gemm(rows, M, ne0 // 256) for M in range(1, 513) for rows, ne0 in ((QR, E), (E, AH), (F, E), (E, F), (V, E)))
    buffers += part(512, 64, 8, 128, 2 ** 31 - 1)
    assert buffers <= fixed - weights <= buffers + 256 * 4 * V + (110 << 20)
