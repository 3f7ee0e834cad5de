"""Small batches at ModernBERT-base size against the CPU oracle, with the
total token count T swept across the small-M GEMM's tile rules (every
projection runs the whole-K kernel up to 128 rows: 32-row tiles while the
grid fits one workgroup per CU, 64-row tiles past it; Wi + GeGLU on 32- or
64-column tiles by the same rule), the split counts of the residual GEMMs
(Wo / MlpWo split over K into 2 to 6 parts that the next LayerNorm sums,
fewer parts as T grows) and the forward prologue's 32-token chunks (ragged
sequences, one to three per batch, independent and plain).

Bars as in test_gpu_forward: fp32 max |dp| <= 1e-5 and logits within
1e-4 * (1 + |logit|); bf16 and fp16 max |dp| <= 2e-3; argmax agreement
(16-bit modes: on every request whose oracle top-two probabilities are more
than 4e-3 apart)."""
import numpy as np
import pytest

import oracle
from test_gpu_forward import WORKERS, compare

pytestmark = pytest.mark.gpu

# T values on both sides of the boundaries: 32 / 64 / 96 / 128 rows, and
# the grid sizes (N / 32) * ceil(T / 32) around 256 workgroups for N = 2304.
TOTALS = [9, 31, 33, 63, 64, 65, 96, 97, 112, 127, 128]


def batch_with_total(total, vocab, rng):
    """One to three packed requests whose lengths add up to `total`."""
    from decide_amd.nn import build_sequence
    from decide_amd.synth import MASK_ID, pack_request

    nseq = int(rng.integers(1, min(3, total // 9) + 1))
    # each sequence at least 9 tokens, the rest spread at random
    lens = 9 + rng.multinomial(total - 9 * nseq, [1.0 / nseq] * nseq)
    batch = []
    for i, n in enumerate(lens):
        k = int(rng.integers(1, min(4, (n - 3) // 2) + 1))  # options, each at least 2 tokens
        premise = int(rng.integers(3, n - 2 * k + 1))  # [CLS] ... [SEP], at least 3 tokens
        rest = n - premise
        opt = [2] * k
        for j in range(rest - 2 * k):
            opt[j % k] += 1
        ids = pack_request(rng, premise, opt, vocab)
        assert len(ids) == n
        batch.append(build_sequence(ids, MASK_ID, independent=bool(i % 2 == 0)))
    return batch


@pytest.fixture(scope="module")
def base_small():
    from decide_amd import Engine, NoGPUError, modernbert_base
    from decide_amd.synth import random_weights

    cfg = modernbert_base()
    w = random_weights(cfg, seed=3)
    try:
        engs = {p: Engine(cfg, w, precision=p) for p in ("fp32", "bf16", "fp16")}
    except NoGPUError:
        pytest.skip("no GPU")
    yield cfg, oracle.OracleModel(cfg, w), engs
    for e in engs.values():
        e.close()


@pytest.mark.parametrize("total", TOTALS)
def test_small_batch_matches_oracle(base_small, total):
    cfg, orc, engs = base_small
    rng = np.random.default_rng(1000 + total)
    batch = batch_with_total(total, cfg.vocab, rng)
    assert sum(len(s.ids) for s in batch) == total
    oracle.set_workers(WORKERS)
    want = orc.forward(batch)
    for prec in ("fp32", "bf16", "fp16"):
        compare(engs[prec].forward(batch), want, batch, prec)


@pytest.mark.parametrize("prec", ["bf16", "fp16"])
def test_small_m_operand_paths_agree(base_small, prec):
    """dn_set_small_m_loads: the small-M GEMM's two operand paths (whole rows
    through LDS by global->LDS DMA, the default; fragments straight into
    registers) feed the MFMAs the same operands in the same order, so every
    batch size gives bit-identical logits."""
    cfg, _, engs = base_small
    eng = engs[prec]
    rng = np.random.default_rng(77)
    try:
        for total in TOTALS:
            batch = batch_with_total(total, cfg.vocab, rng)
            eng.set_small_m_loads(1)
            lds = eng.forward(batch)
            eng.set_small_m_loads(0)
            regs = eng.forward(batch)
            assert np.array_equal(lds, regs), (total, float(np.max(np.abs(lds - regs))))
    finally:
        eng.set_small_m_loads(1)


@pytest.mark.parametrize("total", [129, 256, 257, 897, 1000, 1024, 1345])
def test_folded_small_batch_matches_oracle(base_small, total):
    """Batches above the small-M kernels (129 tokens up) on both sides of the
    folded GEMMs' tile rules: attn_norm and mlp_norm run inside the GEMMs around
    them, statistics in 64-column parts (fp16: above 1,024 tokens). With the switch
    off the LayerNorm kernels run: other roundings, the same bars."""
    cfg, orc, engs = base_small
    rng = np.random.default_rng(2000 + total)
    batch = batch_with_total(total, cfg.vocab, rng)
    oracle.set_workers(WORKERS)
    want = orc.forward(batch)
    for prec in ("bf16", "fp16"):
        got = engs[prec].forward(batch)
        compare(got, want, batch, prec)
        try:
            engs[prec].set_ln_fold(False)
            plain = engs[prec].forward(batch)
            assert np.array_equal(plain, got) == (prec == "fp16" and total <= 1024)
            compare(plain, want, batch, prec)
            compare(got, plain.astype(np.float64), batch, prec)
        finally:
            engs[prec].set_ln_fold(True)


@pytest.mark.parametrize("total", [129, 300, 1024])
def test_fp16_outlier_channel(total):
    """A channel whose residual values (up to ~1,000) times its mlp_norm weight (300)
    leave fp16's range, while the normalised row times the weight stays under
    sqrt(768) x 300 = 8,314: fp16 forwards of a single request's size normalise
    first and stay at the 16-bit bar. The projections' weights of the channel are
    1/300 of the others', so it weighs like them."""
    from decide_amd import Engine
    from decide_amd.nn import Config
    from decide_amd.synth import random_weights

    cfg = Config(hidden=768, intermediate=1152, heads=12, layers=3, vocab=50368, half_window=64,
                 layer_types=["full_attention", "sliding_attention", "full_attention"])
    w = random_weights(cfg, seed=11)
    w["model.embeddings.norm.weight"][100] = 300.0
    w["model.layers.0.attn.Wqkv.weight"][:, 100] /= 300.0
    for i in range(cfg.layers):
        w[f"model.layers.{i}.mlp_norm.weight"][100] = 300.0
        w[f"model.layers.{i}.mlp.Wi.weight"][:, 100] /= 300.0
    batch = batch_with_total(total, cfg.vocab, np.random.default_rng(total))
    oracle.set_workers(WORKERS)
    want = oracle.OracleModel(cfg, w).forward(batch)
    with Engine(cfg, w, precision="fp16") as eng:
        compare(eng.forward(batch), want, batch, "fp16")


@pytest.mark.parametrize("prec,lens", [("bf16", (31,)), ("fp32", (32, 33)), ("bf16", (257, 225, 30)),
                                       ("fp16", (1024,)), ("bf16", (1025,)), ("fp32", (2048,)), ("fp32", (2049,))])
def test_key_split_attention_matches_oracle(base_small, prec, lens):
    """Attention with each query chunk's keys split over a workgroup's waves:
    sequences of one unit (32 keys), ragged last units and chunks, more units
    than waves, and both sides of the item limits (1,024 tokens in 16 bits, 2,048
    in fp32). Independent options and plain sequences."""
    from decide_amd.nn import build_sequence
    from decide_amd.synth import MASK_ID, pack_request

    cfg, orc, engs = base_small
    rng = np.random.default_rng(sum(lens))
    batch = [build_sequence(pack_request(rng, n - 3 * 5, [5] * 3, cfg.vocab), MASK_ID, independent=i % 2 == 0)
             for i, n in enumerate(lens)]
    oracle.set_workers(WORKERS)
    compare(engs[prec].forward(batch), orc.forward(batch), batch, prec)


@pytest.mark.parametrize("prec,tokens", [("bf16", 768), ("bf16", 769), ("fp32", 1536), ("fp32", 1537)])
def test_key_split_line_follows_heads(prec, tokens):
    """The key-split attention's line is in (work item, head) pairs too: at 16 heads
    6 items in 16 bits and 12 in fp32. Both sides against the oracle."""
    from decide_amd import Engine
    from decide_amd.nn import Config, build_sequence
    from decide_amd.synth import MASK_ID, pack_request, random_weights

    cfg = Config(hidden=1024, intermediate=512, heads=16, layers=2, vocab=50368, half_window=64,
                 layer_types=["full_attention", "sliding_attention"])
    w = random_weights(cfg, seed=12)
    batch = [build_sequence(pack_request(np.random.default_rng(tokens), tokens - 15, [5] * 3, cfg.vocab), MASK_ID, True)]
    oracle.set_workers(WORKERS)
    with Engine(cfg, w, precision=prec) as eng:
        compare(eng.forward(batch), oracle.OracleModel(cfg, w).forward(batch), batch, prec)


def test_captured_forward_follows_new_weights():
    """A captured dn_forward_device of a batch that folds the LayerNorm (300 tokens
    in bf16): every replay gives the eager logits, and after an upload of other
    weights the replays give theirs, the folded column sums among them. The
    program's own eager forwards run between the replays."""
    import torch

    from decide_amd import Engine
    from decide_amd.nn import Config, flatten, row_tokens
    from decide_amd.synth import random_weights

    cfg = Config(hidden=768, intermediate=1152, heads=12, layers=3, vocab=50368, half_window=64,
                 layer_types=["full_attention", "sliding_attention", "full_attention"])
    w, w2 = random_weights(cfg, seed=1), random_weights(cfg, seed=2)
    batch = batch_with_total(300, cfg.vocab, np.random.default_rng(5))
    seq_len, ids, pos, opt, _, _ = flatten(batch)
    rows = row_tokens(batch)
    ids, pos, opt, rows = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (ids, pos, opt, rows))
    out = torch.zeros(len(rows), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with Engine(cfg, w, precision="bf16") as eng:
        eng.set_stream(s.cuda_stream)

        def forward():
            eng.forward_device(seq_len, ids.data_ptr(), pos.data_ptr(), opt.data_ptr(), len(rows), rows.data_ptr(),
                               out.data_ptr())

        def eager():
            forward()
            eng.synchronize()
            return out.cpu().numpy()

        def replay():
            out.fill_(7.0)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            return out.cpu().numpy()

        first = eager()
        with torch.cuda.graph(g, stream=s):
            forward()
        for _ in range(3):
            assert np.array_equal(replay(), first)
            assert np.array_equal(eager(), first)
        eng.load(w2)
        second = [replay() for _ in range(2)]
        want = eager()
        assert not np.array_equal(want, first)
        for got in second + [replay()]:
            assert np.array_equal(got, want)
