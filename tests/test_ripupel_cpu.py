"""Ripupel on the CPU reference ops: reading a checkpoint folder, and the engine's, cache's, state
slots' and scheduler's part in it (portions, mixed batches, reuse, generation) against the plain
implementation of ripupel_oracle.py.  The GPU kernels have the same tests in test_ripupel_gpu.py."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import ripupel_oracle as O
from voice_enabled_browser_automation_amd import ops
from voice_enabled_browser_automation_amd.models import model_class
from voice_enabled_browser_automation_amd.models.config import LatentAttentionConfig, MoEConfig, RipupelConfig, config_from_dir, get_config
from voice_enabled_browser_automation_amd.models.ripupel import RipupelModel
from voice_enabled_browser_automation_amd.ops import mixers
from voice_enabled_browser_automation_amd.runtime.engine import LLMEngine
from voice_enabled_browser_automation_amd.runtime.kv_cache import CacheLayer, PagedKVCache
from voice_enabled_browser_automation_amd.runtime.scheduler import TokenScheduler
from voice_enabled_browser_automation_amd.runtime.weights import load_llm

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# unequal layers: odd sizes, blocks that need padding, a layer without a feed-forward, one expert of several and
# several, a latent shared by two later layers, a convolution of one tap
CFG = O.model_config(76, 101, [
    O.latent_layer(3, 20, 6, 24, 40, O.moe(5, 2, 24)),
    O.rglru_layer(60, 3, 4, O.dense(56)),
    O.latent_layer(5, 12, 6, 8, 40, None, scale=0.3, kv_from=0),
    O.rglru_layer(40, 1, 1, O.moe(4, 1, 40)),
    O.latent_layer(1, 32, 10, 16, 33, O.dense(33), base=500.0),
    O.latent_layer(2, 16, 6, 16, 40, O.moe(3, 3, 16), kv_from=0),
], eps=1e-3)


def tokens(n, seed, vocab=101):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


@pytest.fixture(scope="module")
def folder(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("ripupel") / "m")
    O.save_model(d, CFG, O.random_weights(CFG, 5))
    return d


@pytest.fixture(scope="module")
def weights():
    return O.random_weights(CFG, 5)


@pytest.fixture(scope="module")
def model(folder):
    return load_llm(folder, device="cpu", dtype=torch.float32)


def engine(model, **kw):
    return LLMEngine(model, **dict(dict(max_seqs=3, max_model_len=256, kv_blocks=40), **kw))


@pytest.mark.parametrize("rows", [1, 7, 16, 17, 777])
def test_branch_rows_of_prompts(rows):
    """A row of the branch buffer for each of a token's experts, and four for each of few tokens (a 32-bit product's quarters): not four
    for every token of a prompt."""
    top = 2
    cfg = O.model_config(76, 101, [O.rglru_layer(60, 3, 4, O.dense(56)), O.rglru_layer(40, 1, 1, O.moe(4, top, 40))])
    w = O.random_weights(cfg, 5)
    for dtype, few in ((torch.float32, 4 * min(rows, 16)), (torch.bfloat16, 0)):
        m = RipupelModel(RipupelConfig.from_json(cfg), weights=w, dtype=dtype)
        assert m.row_buffers(rows, 256)["branch"].shape[0] == max(top * rows, few)


def test_config_and_registry(folder):
    cfg = config_from_dir(folder)
    assert isinstance(cfg, RipupelConfig) and get_config(folder) == cfg and model_class(cfg) is RipupelModel
    assert cfg.vocab_size == 101 and cfg.hidden == 76 and cfg.n_layers == 6 and cfg.norm_eps == 1e-3 and cfg.embed_scale == 0.7
    a = cfg.layers[2].mixer
    assert a == LatentAttentionConfig(heads=5, dim=12, rot_dim=6, vdim=8, kv_rank=40, scale=0.3, rot_base=10000.0, kv_from=0)
    assert cfg.layers[2].mlp is None and cfg.layers[0].mlp == MoEConfig(experts=5, top=2, ff=24)
    assert cfg.layers[1].mixer.block == 20 and cfg.layers[3].mixer.conv == 1
    assert model_class(get_config("ripupel-tiny")) is RipupelModel


@pytest.mark.parametrize("change", [
    lambda j: j["layers"][0].update(type="parallel"),
    lambda j: j["layers"][1]["mlp"].update(kind="routed"),
    lambda j: j["layers"][1]["mixer"].update(blocks=7),
    lambda j: j["layers"][1]["mixer"].update(conv=0),
    lambda j: j["layers"][0]["mixer"]["rot"].update(dims=4),
    lambda j: j["layers"][0]["mixer"].update(rot_dim=7),
    lambda j: j["layers"][0]["mlp"]["router"].update(top=6),
    lambda j: j["layers"][2]["mixer"].update(kv_from=1),
    lambda j: j["layers"][2]["mixer"].update(kv_from=4),
    lambda j: j["layers"][5]["mixer"].update(kv_from=2),
    lambda j: j["layers"][2]["mixer"].update(kv_rank=41),
    lambda j: j["layers"][2]["mixer"]["rot"].update(base=20000.0),
])
def test_config_refuses_what_it_does_not_know(change):
    j = json.loads(json.dumps(CFG))
    RipupelConfig.from_json(j)
    change(j)
    with pytest.raises(ValueError):
        RipupelConfig.from_json(j)


@pytest.mark.parametrize("name", ["scale", "kv_rank", "heads"])
def test_missing_constants_are_errors(name):
    j = json.loads(json.dumps(CFG))
    del j["layers"][0]["mixer"][name]
    with pytest.raises(KeyError):
        RipupelConfig.from_json(j)


@pytest.mark.parametrize("name", ["l0.mix.q", "l1.mix.ra", "l1.mix.lam", "l0.mlp.router", "l0.mlp.e1.down", "l4.mix.dkv.norm", "embed"])
def test_wrong_tensor_shape_is_an_error(weights, name):
    w = dict(weights)
    w[name] = w[name][:-1]
    with pytest.raises(ValueError):
        RipupelModel(RipupelConfig.from_json(CFG), weights=w, dtype=torch.float32)


def test_whole_prompt_and_layers(model, weights):
    t = tokens(90, 1)
    want, res = O.forward(CFG, weights, t, layers=True)
    eng = engine(model)
    seq = eng.new_sequence([])
    seen = []
    run = model._layer
    model._layer = lambda li, bufs, M, kv, x, *a: (run(li, bufs, M, kv, x, *a), seen.append(x[:, :76].clone()))
    try:
        got = eng.step_batch([(seq, t)], range(len(t)))
    finally:
        del model._layer
    for g, r in zip(seen, res):
        assert torch.allclose(g.double(), r, atol=2e-4)
    assert O.logit_error(got, want).max() < 1e-5


@pytest.mark.parametrize("cuts", [[2], [1], [16], [17, 3], [70, 2]])
def test_portions(model, weights, cuts):
    t = tokens(83, 2)
    want = O.forward(CFG, weights, t)
    eng = engine(model)
    seq, out, i, k = eng.new_sequence([]), [], 0, 0
    while i < len(t):
        part = t[i : i + cuts[k % len(cuts)]]
        out.append(eng.step_batch([(seq, part)], range(len(part))).clone())
        i, k = i + len(part), k + 1
    assert O.logit_error(torch.cat(out), want).max() < 1e-5


def test_mixed_batches_and_reuse(model, weights):
    """Unequal requests in common steps (one skipping steps), pages and slots given back and used again,
    against every request alone; the pool is exactly as large as the live requests need."""
    eng = engine(model, kv_blocks=1 + 3 * 6)
    reqs = {n: tokens(n, n) for n in (95, 41, 7, 64, 88, 1)}
    want = {n: O.forward(CFG, weights, t) for n, t in reqs.items()}
    live, queue, at, got, rng = {}, list(reqs), {}, {n: [] for n in reqs}, np.random.default_rng(0)
    used_sids = []
    while queue or live:
        while queue and len(live) < 3:
            n = queue.pop(0)
            live[n], at[n] = eng.new_sequence([]), 0
            used_sids.append(live[n].sid)
        entries = []
        for n, seq in live.items():
            if rng.random() < 0.25 and len(live) > 1:
                continue
            k = int(rng.choice([1, 1, 2, 5, 17, 40]))
            entries.append((n, reqs[n][at[n] : at[n] + k]))
        if not entries:
            continue
        lg = eng.step_batch([(live[n], p) for n, p in entries], range(sum(len(p) for _, p in entries)))
        i = 0
        for n, p in entries:
            got[n].append(lg[i : i + len(p)].clone())
            i += len(p)
            at[n] += len(p)
        for n in [n for n, _ in entries if at[n] == n]:
            eng.free_sequence(live.pop(n))
    assert len(set(used_sids)) == 3 and len(used_sids) == 6
    for n in reqs:
        assert O.logit_error(torch.cat(got[n]), want[n]).max() < 1e-5, n
    assert eng.blocks.n_free() == 18


def test_one_planted_mistake_per_mechanism_shows(weights):
    """The comparisons are sharp: the oracle with one mechanism slightly wrong differs by far more than
    the tolerance used above."""
    t = tokens(60, 3)
    want = O.forward(CFG, weights, t)

    def changed(f):
        w = {k: v.clone() for k, v in weights.items()}
        c = json.loads(json.dumps(CFG))
        f(c, w)
        return O.logit_error(O.forward(c, w, t), want).max()

    def each(w, end, f):
        for k in w:
            if k.endswith(end):
                w[k] = f(w[k])

    faults = {
        "sink left out": lambda c, w: each(w, "sink", lambda v: v - 40),
        "gate left out": lambda c, w: each(w, "mix.g", lambda v: v * 0),
        "conv one tap late": lambda c, w: each(w, "mix.conv", lambda v: v.roll(1, -1)),
        "gelu branch bias": lambda c, w: each(w, "y.b", lambda v: v * 0),
        "decay": lambda c, w: each(w, "lam", lambda v: v + 0.1),
        "gates swapped": lambda c, w: [w.update({p + "ra": w[p + "ri"], p + "ri": w[p + "ra"]}) for p in ("l1.mix.", "l3.mix.")],
        "latent norm": lambda c, w: each(w, "dkv.norm", lambda v: v * 0 + 1),
        "rotation base": lambda c, w: [L["mixer"]["rot"].update(base=9000.0) for L in c["layers"] if "rot" in L["mixer"]],
        "embedding scale": lambda c, w: c["embedding"].update(scale=0.72),
        "wrong layer's latent": lambda c, w: (c["layers"][2]["mixer"].pop("kv_from"), w.update(
            {"l2.mix.dkv": w["l0.mix.dkv"], "l2.mix.dkv.norm": w["l0.mix.dkv.norm"]})),
        "one expert fewer": lambda c, w: c["layers"][0]["mlp"]["router"].update(top=1),
    }
    for name, f in faults.items():
        assert changed(f) > 1e-3, name


def test_state_starts_from_zero_in_a_used_slot(model, weights):
    eng = engine(model, max_seqs=1)
    for seed in (11, 12):
        t = tokens(30, seed)
        seq = eng.new_sequence([])
        got = eng.step_batch([(seq, t)], range(len(t)))
        assert O.logit_error(got, O.forward(CFG, weights, t)).max() < 1e-5
        eng.free_sequence(seq)
    assert all(s.abs().max() > 0 for s in eng.kv.state if s.numel())


def test_prefix_cache_only_without_recurrent_layers(model):
    """Blocks alone cannot resume a recurrent state; a stack of attention layers alone is served from them."""
    t = tokens(64, 4)
    eng = engine(model)
    for _ in range(2):
        seq = eng.new_sequence(t)
        assert seq.n_computed == 0
        eng.prefill(seq)
        eng.free_sequence(seq)
    assert eng.blocks.n_free() == eng.blocks.num_blocks - 1 and not eng.blocks.cache
    cfg = O.model_config(76, 101, [O.latent_layer(3, 20, 6, 24, 40, O.dense(32)), O.latent_layer(2, 16, 6, 16, 40, None, kv_from=0)])
    w = O.random_weights(cfg, 2)
    eng = engine(RipupelModel(RipupelConfig.from_json(cfg), weights=w, dtype=torch.float32))
    want = O.forward(cfg, w, t)[-1:]
    for cached in (0, 48):
        seq = eng.new_sequence(t)
        assert seq.n_computed == cached
        assert O.logit_error(eng.prefill(seq), want).max() < 1e-5
        eng.free_sequence(seq)


def test_a_stack_without_attention(model):
    cfg = O.model_config(64, 50, [O.rglru_layer(48, 2, 3, O.dense(32)), O.rglru_layer(32, 1, 2, None)])
    w = O.random_weights(cfg, 3)
    eng = LLMEngine(RipupelModel(RipupelConfig.from_json(cfg), weights=w, dtype=torch.float32), max_seqs=2, max_model_len=128)
    t = tokens(100, 1, 50)
    seq = eng.new_sequence([])
    got = torch.cat([eng.step_batch([(seq, t[i : i + 70])], range(len(t[i : i + 70]))).clone() for i in (0, 70)])
    assert O.logit_error(got, O.forward(cfg, w, t)).max() < 1e-5


def test_engine_prefill_paths_agree(model, weights):
    t = tokens(150, 6)
    want = O.forward(CFG, weights, t)
    eng = engine(model)
    a, b = eng.new_sequence(t), eng.new_sequence(t)
    assert O.logit_error(eng.prefill(a, chunk=100), want[-1:]).max() < 1e-5
    eng.prefill_batch([(b, len(t) - 1)])
    got = eng.run_rows([(b, t[-1])])
    assert O.logit_error(got, want[-1:]).max() < 1e-5


def greedy(cfg, weights, prompt, n):
    t = list(prompt)
    for _ in range(n):
        t.append(int(O.forward(cfg, weights, t)[-1].argmax()))
    return t[len(prompt):]


def test_greedy_generation_through_the_scheduler(model, weights):
    prompts = [tokens(n, 20 + n) for n in (37, 3, 70, 1, 18)]
    eng = engine(model, max_seqs=2)
    sched = TokenScheduler(eng, token_budget=24)
    outs = sched.generate(prompts, 6)
    assert outs == [greedy(CFG, weights, p, 6) for p in prompts]
    assert sched.stats["rows"] == sum(len(p) + 5 for p in prompts)
    # a stop token ends a request
    assert sched.generate([prompts[0]], 6, stop_ids=[outs[0][1]])[0] == outs[0][: outs[0].index(outs[0][1]) + 1]


def test_cache_layers_share_pages(model):
    layers = [CacheLayer(n_kv_heads=1, k_dim=96), CacheLayer(state=48), CacheLayer(n_kv_heads=1, k_dim=96, shared=0)]
    kv = PagedKVCache.from_layers(layers, 16, 5, 3, dtype=torch.float32)
    assert kv.k[0].shape == (5, 1, 16, 96) and kv.k[2] is kv.k[0] and kv.state[1].shape == (3, 48) and kv.k[1].numel() == 0
    assert PagedKVCache.layer_bytes_per_block(layers, 16) == 2 * 16 * 96
    kv = engine(model).kv
    assert kv.k[2] is kv.k[0] and kv.k[5] is kv.k[0] and kv.k[4] is not kv.k[0]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_weight_layouts(dtype):
    """Fragment order and tiles name every element once, where the kernels look for it."""
    epl = 16 // dtype.itemsize
    N, K = 48, 128
    w = torch.arange(N * K).view(N, K).remainder(251).to(dtype)
    f = ops.fragments(w).view(N // 16, K // (4 * epl), 64, epl)
    for T, s, lane, e in ((0, 0, 0, 0), (1, 2, 37, 3), (2, K // (4 * epl) - 1, 63, epl - 1)):
        assert f[T, s, lane, e] == w[16 * T + lane % 16, 4 * epl * s + epl * (lane // 16) + e]
    t = ops.tile_weights(w[None])[0]
    if dtype == torch.bfloat16:
        assert torch.equal(t, ops.tile_weight(w))
    t = t.reshape(N // 16, K // (16 * epl), 4, 64, epl)
    for T, kg, s, lane, e in ((0, 0, 1, 5, 1), (2, K // (16 * epl) - 1, 3, 63, 2)):
        assert t[T, kg, s, lane, e] == w[16 * T + lane % 16, 16 * epl * kg + 4 * epl * (lane // 16) + epl * s + e]
    g = torch.arange(2 * 2 * 32 * 32).view(2, 2, 32, 32).remainder(251).to(dtype)
    f = ops.gate_fragments(g).view(2, 2, 2, 32 // (4 * epl), 64, epl)
    assert f[1, 1, 0, 0, 33, 1] == g[1, 0, 16 + 33 % 16, epl * (33 // 16) + 1]


def test_launch_sizes():
    assert mixers.latent_chunks(1, 16, 1536) == 24 and mixers.latent_chunks(64, 16, 1536) == 8
    assert mixers.latent_chunks(64, 128, 100000) == 1 and mixers.latent_chunks(1, 1, 1) == 1
    for pairs, E, tile in ((1, 8, 16), (64, 8, 16), (4096, 16, 128), (5, 3, 16)):
        worst = 0
        for heavy in range(pairs + 1):                 # the other pairs spread one by one
            rest = min(pairs - heavy, E - 1)
            worst = max(worst, -(-heavy // tile) + rest)
        assert mixers.moe_tiles(pairs, E, tile) >= worst


def test_trace_replay_command(folder, weights, tmp_path):
    """bin/trace_run end to end on the reference ops: two requests in common steps, wanted logits in order."""
    a, b = tokens(70, 31), tokens(20, 32)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:69], "want": [0, 68]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": a[69:], "want": []}, {"id": "b", "tokens": b[:2], "want": []}],
              "end": ["a"]},
             {"step": 2, "entries": [{"id": "b", "tokens": b[2:], "want": [17, 3]}], "end": ["b"]}]
    out = tmp_path / "out"
    r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", folder, "--dtype", "float32", "--out", str(out),
                        "--max-tokens", "128", "--device", "cpu"], input="".join(json.dumps(s) + "\n" for s in steps),
                       capture_output=True, text=True, timeout=300, env=dict(os.environ, PYTHONDONTWRITEBYTECODE="1"))
    assert r.returncode == 0, r.stderr[-2000:]
    assert [x for x in r.stdout.split("\n") if x] == ["done 0", "done 1", "done 2"]
    wa, wb = O.forward(CFG, weights, a), O.forward(CFG, weights, b)
    read = lambda n: torch.from_numpy(np.fromfile(out / f"{n}.f32", dtype="<f4")).view(-1, 101)  # noqa: E731
    assert O.logit_error(read(0), wa[[0, 68]]).max() < 1e-5
    assert not (out / "1.f32").exists()
    assert O.logit_error(read(2), wb[[19, 5]]).max() < 1e-5


def test_generate_command(folder, weights):
    r = subprocess.run([sys.executable, "-m", "voice_enabled_browser_automation_amd.generate", "--model", folder, "--ids",
                        "5,6,7", "--ids", "9", "--max-new", "3", "--dtype", "float32", "--device", "cpu", "--max-model-len",
                        "64"], capture_output=True, text=True, timeout=300, cwd=ROOT)
    assert r.returncode == 0, r.stderr[-2000:]
    got = [json.loads(x)["tokens"] for x in r.stdout.split("\n") if x]
    assert got == [greedy(CFG, weights, p, 3) for p in ([5, 6, 7], [9])]


def test_intent_engine_serves_a_ripupel_preset():
    """The grammar-constrained intent scheduler runs it like its other models."""
    from voice_enabled_browser_automation_amd.brain.intent_engine import LLMIntentEngine
    from voice_enabled_browser_automation_amd.contracts import ParseResponse, safe_parse
    from voice_enabled_browser_automation_amd.tokenizer import load_tokenizer

    m = load_llm("ripupel-tiny", device="cpu")
    eng = LLMEngine(m, max_seqs=2, max_model_len=2048)
    brain = LLMIntentEngine(eng, load_tokenizer("llama3"), budget_chars=160)
    out = brain.parse({"text": "scroll down", "context": {}})
    assert safe_parse(ParseResponse, out).success
