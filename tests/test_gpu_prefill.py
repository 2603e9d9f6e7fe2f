"""GPU parity of the batched prompt (pio_qwen3_prefill): a prompt's positions
in one pass per layer -- every int8 linear once over all rows on the W8 MFMA
GEMM, causal attention and KV-cache rows for every position -- as the
reference forwards the whole prompt at its first step
(ip/models/qwen3_0_6b/architecture.py:204-213).

Bars, as for the step decoder (tests/test_gpu_decode.py): logits against the
float64 oracle (qwen3_ref.forward_all, evaluated in one batched pass) within
max(1e-4, 4x numpy-fp32's own error) of the logit rms, argmax agreement
wherever the oracle's top-2 gap is clear; fp16 KV as there. The decode steps
that follow a batched prompt read the cache it wrote, so their logits are held
to the same bar on the GPU's own ids."""
import sys

import numpy as np
import pytest

from oracle import qwen3_ref
from tests.test_gpu_decode import _assert_logit_bar, _check_argmax

pytestmark = pytest.mark.gpu


def _say(m):
    print(m, flush=True)
    sys.stdout.flush()


def _against_oracle(got, ids, pos, rcfg, w, what):
    seq = np.asarray(ids[:max(pos) + 1])
    e64 = qwen3_ref.forward_all(rcfg, w, seq, pos, np.float64)
    e32 = qwen3_ref.forward_all(rcfg, w, seq, pos, np.float32).astype(np.float64)
    errs, errs32 = [], []
    for i, p in enumerate(pos):
        rms = float(np.sqrt(np.mean(e64[i] * e64[i])))
        errs.append(float(np.abs(got[i] - e64[i]).max()) / rms)
        errs32.append(float(np.abs(e32[i] - e64[i]).max()) / rms)
        _say(f"{what}: position {p}: err {errs[-1]:.2e} (numpy fp32 {errs32[-1]:.2e})")
        _check_argmax(got[i:i + 1], e64[i:i + 1], 1e-3)
    _assert_logit_bar(errs, errs32, rcfg, what)


def _small(**over):
    from mod_amd.qwen3 import Qwen3Config
    kw = dict(n_layers=2, hidden=1024, n_heads=16, n_kv_heads=8, head_dim=128, intermediate=3072,
              vocab=1000, max_seq=256)
    kw.update(over)
    return Qwen3Config(**kw), qwen3_ref.Qwen3Config(**kw)


@pytest.mark.parametrize("kv_dtype", ["float32", "float16"])
def test_prefill_last_logits_and_chunks(torch_dev, kv_dtype):
    """A 70-token prompt in one batch: the last position's logits against the
    oracle; the same prompt in three batches (31 + 1 + 38 positions: the
    second starts from the first one's cache) gives the same logits to fp32
    rounding; and the next id is the argmax, as the step would write it."""
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, rcfg = _small(kv_dtype=kv_dtype)
    w = random_weights(cfg, seed=61)
    dec = Qwen3Int8Decoder(cfg, w)
    P = 70
    prompt = np.random.default_rng(62).integers(0, cfg.vocab, size=P).astype(np.int32)
    dec.reset(prompt)
    dec.prefill(P, logits=True)
    ids, one = dec.read(P + 1, with_logits=True)
    assert np.array_equal(ids[:P], prompt)
    assert int(ids[P]) == int(np.argmax(one))
    _against_oracle(one[None], prompt, [P - 1], rcfg, w, f"prefill last logits ({kv_dtype} KV)")
    dec.reset(prompt)
    dec.prefill(31)
    dec.prefill(1)
    dec.prefill(P - 32, logits=True)
    _, three = dec.read(0, with_logits=True)
    rms = float(np.sqrt(np.mean(one.astype(np.float64) ** 2)))
    diff = float(np.abs(three - one).max()) / rms
    _say(f"one batch vs three: max diff {diff:.2e} x rms")
    assert diff <= (1e-4 if kv_dtype == "float32" else 2e-3), diff


@pytest.mark.parametrize("P,intermediate", [(385, 3072), (421, 3136), (512, 3072)])
def test_prefill_long_batch(torch_dev, P, intermediate):
    """From 385 rows the gate_up GEMM's epilogue forms silu(g) * u (row tiles of
    1, 37 and 128 rows at the end): logits against the oracle, and against the
    same prompt in batches of at most 100, whose SwiGLU is a kernel of its own
    (the bar of the test above: fp32 rounding in another order)."""
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, rcfg = _small(max_seq=512, intermediate=intermediate)
    w = random_weights(cfg, seed=63)
    dec = Qwen3Int8Decoder(cfg, w)
    prompt = np.random.default_rng(64).integers(0, cfg.vocab, size=P).astype(np.int32)
    _say(f"prefill long batch P={P} I={intermediate}")
    dec.reset(prompt)
    dec.prefill(P, logits=True)
    one = dec.read(0, with_logits=True)[1].copy()
    _against_oracle(one[None], prompt, [P - 1], rcfg, w, f"prefill of {P}")
    dec.reset(prompt)
    for a in range(0, P, 100):
        dec.prefill(min(100, P - a), logits=a + 100 >= P)
    parts = dec.read(0, with_logits=True)[1]
    diff = float(np.abs(parts - one).max()) / float(np.sqrt(np.mean(one.astype(np.float64) ** 2)))
    _say(f"one batch vs parts: max diff {diff:.2e} x rms")
    assert diff <= 1e-4, diff


def _cache(torch, dec, cfg):
    """Views of the decoder's K and V cache, [layer][kv head][position][slot]:
    they follow the logits in its memory, each region padded to 256 bytes."""
    from mod_amd.ops import lib
    typ, size = ("<f4", 4) if cfg.kv_dtype == "float32" else ("<f2", 2)
    shape = (cfg.n_layers, cfg.n_kv_heads, cfg.max_seq, cfg.head_dim)

    def pad(n):
        return (n + 255) // 256 * 256

    class At:
        def __init__(self, p):
            self.__cuda_array_interface__ = {"shape": shape, "typestr": typ, "data": (p, False), "version": 2}

    k = lib.pio_qwen3_logits(dec._h) + pad(4 * cfg.vocab)
    return [torch.as_tensor(At(p), device="cuda:0") for p in (k, k + pad(int(np.prod(shape)) * size))]


@pytest.mark.parametrize("kv_dtype", ["float32", "float16"])
@pytest.mark.parametrize("P,at", [(100, 70), (300, 283), (40, 31)])
def test_prefill_value_of_inf_stays_behind_its_position(torch_dev, kv_dtype, P, at):
    """A token whose value row holds an inf (past the range of the cache's type)
    leaves the positions before it as they are without it: the second layer's
    keys and values, which carry the first one's attention. The batches keep the
    keys of a workgroup whole (100, 40) and split them (300)."""
    import torch
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, _ = _small(max_seq=320, kv_dtype=kv_dtype)
    w = random_weights(cfg, seed=65)
    w["embed"] = w["embed"].copy()
    L = w["layers"][0]
    row = (cfg.n_heads + cfg.n_kv_heads) * 128 + 3        # value dim 3 of kv head 0
    w["embed"][7] = L["w_qkv"][row]                       # aligned with token 7: about 7 times any other's
    top = np.sqrt(cfg.hidden * float((L["w_qkv"][row].astype(np.float64) ** 2).sum()))
    L["s_qkv"][row] = 1.5 * (3.4e38 if kv_dtype == "float32" else 65504.0) / top
    L["b_qkv"][row] = 0
    L["w_o"][:, [3, 131]] = 0                             # that dim of the heads that read it
    dec = Qwen3Int8Decoder(cfg, w)
    prompt = np.random.default_rng(66).integers(8, cfg.vocab, size=P).astype(np.int32)
    _say(f"prefill with a value of inf: {kv_dtype} KV, {P} positions, at {at}")
    rows = []
    for tok in (8, 7):
        prompt[at] = tok
        dec.reset(prompt)
        dec.prefill(P)
        dec.read(0)
        kc, vc = _cache(torch, dec, cfg)
        assert bool(torch.isinf(vc[0, 0, at]).any()) == (tok == 7)
        assert bool(torch.isfinite(vc[0, :, :at]).all())
        rows.append([c[1, :, :at].float().cpu() for c in (kc, vc)])
    for a, b in zip(*rows):
        assert bool(torch.isfinite(b).all())
        # one attention column in another order of sums; fp16 rows may round the other way
        tol = 2e-5 if kv_dtype == "float32" else 2e-3
        assert float((a - b).abs().max()) <= tol * float(a.abs().max())


def test_prefill_fp16_keys_split(torch_dev):
    """fp16 KV where the attention splits its keys over workgroups: a batch of
    300 positions, then a late one of 40, against the oracle and against batches
    of at most 100, the first two of which keep them whole (the bar of the first
    test: fp16 cache rows that round the other way)."""
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, rcfg = _small(max_seq=384, kv_dtype="float16")
    w = random_weights(cfg, seed=69)
    dec = Qwen3Int8Decoder(cfg, w)
    prompt = np.random.default_rng(70).integers(0, cfg.vocab, size=340).astype(np.int32)
    logits = []
    for sizes in ((300, 40), (100, 100, 100, 40)):
        _say(f"fp16 KV, batches of {sizes}")
        dec.reset(prompt)
        for n in sizes[:-1]:
            dec.prefill(n)
        dec.prefill(sizes[-1], logits=True)
        logits.append(dec.read(0, with_logits=True)[1].copy())
        _against_oracle(logits[-1][None], prompt, [339], rcfg, w, f"fp16 KV, batches of {sizes}")
    rms = float(np.sqrt(np.mean(logits[0].astype(np.float64) ** 2)))
    diff = float(np.abs(logits[0] - logits[1]).max()) / rms
    _say(f"max diff {diff:.2e} x rms")
    assert diff <= 2e-3, diff


def test_prefill_refuses_generated_positions(torch_dev):
    from mod_amd.ops import RocmError
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, _ = _small(n_layers=1)
    dec = Qwen3Int8Decoder(cfg, random_weights(cfg, seed=63))
    dec.reset(np.arange(8, dtype=np.int32))
    with pytest.raises(RocmError, match="prompt positions"):
        dec.prefill(9)
    dec.prefill(8)
    with pytest.raises(RocmError, match="prompt positions"):
        dec.prefill(1)


@pytest.mark.parametrize("kv_dtype", ["float32", "float16"])
@pytest.mark.parametrize("n_heads", [8, 16, 32])
def test_prefill_attention_edge(torch_dev, kv_dtype, n_heads):
    """Either side of the 96 keys up to which a batch's attention has a kernel of
    its own, with 1, 2 and 4 query heads per KV head: batches of 96, 97 and 60 +
    37 positions, each against the oracle."""
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, rcfg = _small(kv_dtype=kv_dtype, n_heads=n_heads)
    w = random_weights(cfg, seed=71)
    dec = Qwen3Int8Decoder(cfg, w)
    prompt = np.random.default_rng(72).integers(0, cfg.vocab, size=97).astype(np.int32)
    for sizes in ((96,), (97,), (60, 36), (60, 37)):
        dec.reset(prompt)
        for n in sizes[:-1]:
            dec.prefill(n)
        dec.prefill(sizes[-1], logits=True)
        got = dec.read(0, with_logits=True)[1]
        _against_oracle(got[None], prompt, [sum(sizes) - 1], rcfg, w, f"{n_heads} heads, {kv_dtype} KV, batches of {sizes}")


@pytest.mark.parametrize("intermediate", [3072, 3088])
def test_prefill_memory(torch_dev, intermediate):
    """What a batch of 2048 positions takes from the allocator is no more than its
    activations in fp32 (x, its norm, qkv, the attention's output, [g|u], act),
    with the SwiGLU in the gate_up GEMM (3072) and as a kernel of its own. At this
    size no linear and no attention splits a sum, so nothing else is taken."""
    from mod_amd import ops
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, _ = _small(max_seq=2048, intermediate=intermediate)
    dec = Qwen3Int8Decoder(cfg, random_weights(cfg, seed=67))
    prompt = np.random.default_rng(68).integers(0, cfg.vocab, size=2048).astype(np.int32)
    dec.reset(prompt)
    before = ops.pool_stats()["reserved"]
    dec.prefill(2048)
    dec.read(0)
    taken = ops.pool_stats()["reserved"] - before
    heads, kv = cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim
    row = 4 * (2 * cfg.hidden + (heads + 2 * kv) + heads + 3 * intermediate)
    _say(f"2048 positions, I={intermediate}: {taken} bytes taken, {2048 * row} in fp32")
    assert 0 < taken <= 2048 * row


@pytest.mark.parametrize("mode", ["persistent", "graph"])
def test_prefill_then_decode_small(torch_dev, mode):
    """Prompt in one batch, then greedy steps: the steps' logits (the first
    generated position and every 8th) against the oracle on the GPU's own ids,
    and the ids agree with a run that consumes the prompt step by step."""
    from mod_amd.qwen3 import Qwen3Int8Decoder, random_weights
    cfg, rcfg = _small()
    w = random_weights(cfg, seed=64)
    dec = Qwen3Int8Decoder(cfg, w)
    P, NG = 40, 33
    prompt = np.random.default_rng(65).integers(0, cfg.vocab, size=P).astype(np.int32)
    dec.reset(prompt)
    dec.prefill(P - 1)
    pos, got, done = [], [], 0
    for n in [1] + [8] * 4:
        dec.run(n, mode=mode)
        done += n
        pos.append(P - 2 + done)          # the position the chunk's last step ran
        got.append(dec.read(0, with_logits=True)[1].copy())
    ids = dec.read(P + NG)
    assert np.array_equal(ids[:P], prompt)
    _against_oracle(np.stack(got), ids, pos, rcfg, w, f"prefill + {mode} steps")
    stepwise = dec.generate(prompt, NG, mode=mode)
    match = float(np.mean(stepwise == ids))
    _say(f"batched vs stepwise prompt: token match {match:.2f}")
    assert match >= 0.9


@pytest.mark.parametrize("kv_dtype", ["float32", "float16"])
def test_prefill_c2_generation_vs_oracle(torch_dev, kv_dtype):
    """BASELINE config 2 with the prompt as one batch: 28 layers, vocab
    151936, the 128-token prompt through pio_qwen3_prefill (its last
    position's logits produce the first generated id), then 255 persistent
    steps. The last prompt position's logits and those after every 32nd
    generated token meet the decoder bar against the batched oracle on the
    GPU's own ids, and each read argmax is the id generated next."""
    from mod_amd.qwen3 import Qwen3Config, Qwen3Int8Decoder, random_weights
    P, NG = 128, 256
    cfg = Qwen3Config(max_seq=P + NG, kv_dtype=kv_dtype)
    rcfg = qwen3_ref.Qwen3Config(max_seq=P + NG, kv_dtype=kv_dtype)
    _say("C2 batched prompt: building weights")
    w = random_weights(cfg, seed=0)
    dec = Qwen3Int8Decoder(cfg, w)
    mode = "persistent" if dec.persistent_supported() else "graph"
    prompt = np.random.default_rng(1).integers(0, cfg.vocab, size=P).astype(np.int32)
    dec.reset(prompt)
    dec.prefill(P, logits=True)
    pos = [P - 1]
    logits = [dec.read(0, with_logits=True)[1].copy()]
    done = 1
    for n in [32] * 7 + [31]:
        dec.run(n, mode=mode)
        done += n
        pos.append(P - 2 + done)
        logits.append(dec.read(0, with_logits=True)[1].copy())
    assert done == NG
    ids = dec.read(P + NG)
    assert np.array_equal(ids[:P], prompt)
    for p, lg in zip(pos, logits):
        assert int(np.argmax(lg)) == int(ids[p + 1]), p
    _say("C2 batched prompt: oracle (batched, teacher forced)")
    _against_oracle(np.stack(logits), ids, pos, rcfg, w, f"C2 batched prompt ({kv_dtype} KV)")
