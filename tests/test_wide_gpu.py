"""The wide prefill (prompts of more than one chunk: resident products, the
running-softmax attention past 256 positions, passes of at most 1024 tokens)
against the CPU oracle: logits, greedy tokens and the Peek buffers of the last
chunk, at the edges of its token groups (16, 32), chunks (64), attention
groups and chunks of rows (128), the switch of attention forms (256) and the
passes (1024), with block counts that leave tail blocks and row counts that
leave tiles over, in every weight type and with the binary16 cache."""
import numpy as np
import pytest

from llm_amd import synth
from tests.parity import LOGIT_TOL, cpu_greedy, gpu_generate, greedy_parity, rel_err
from tests.test_model_gpu import _open

pytestmark = pytest.mark.gpu

KINDS = ["attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down"]
SPECS = {
    # 6 and 11 blocks per row (tails of 2 and 3), 20, 12 and 44 tiles, three query heads per KV head
    "tails": lambda: synth.tiny_llama(seed=41, embd=192, heads=3, kv_heads=1, ff=352, ctx=2048),
    "tails-q41": lambda: synth.tiny_llama(seed=42, embd=192, heads=3, kv_heads=1, ff=352, ctx=2048,
                                          types={k: synth.Q4_1 for k in KINDS}),
    "tails-q80": lambda: synth.tiny_qwen(seed=43, embd=320, heads=5, kv_heads=5, ff=416, ctx=2048,
                                         types={k: synth.Q8_0 for k in KINDS}),
    "qwen2": lambda: synth.tiny_qwen(seed=44, ctx=2048),
}


@pytest.mark.parametrize("name,n,f16kv", [
    ("tails", 65, False), ("tails", 96, False), ("tails", 257, False), ("tails", 1024, False), ("tails", 1100, True),
    ("tails-q41", 127, False), ("tails-q41", 300, False), ("tails-q41", 1025, False),
    ("tails-q80", 81, False), ("tails-q80", 383, True), ("qwen2", 128, False), ("qwen2", 256, True),
    ("qwen2", 258, False), ("qwen2", 1087, False)])
def test_wide_prefill(gpu, name, n, f16kv):
    spec = SPECS[name]()
    g, cpu = _open(spec, 1152, f16kv=f16kv)
    L, E, F, kvd = spec.layers, spec.embd, spec.ff, spec.kvd
    prompt = [int(t) for t in synth.prompt(n, n, spec.vocab)]
    logits = g.PrefillLogits(prompt)
    cpu.reset()
    for t in prompt:
        want = cpu.forward(t)
    row = (n - 1) % 64
    tol = 1e-3 if f16kv else 1e-5  # f32 rounding; a K or V at a binary16 tie may round the other way (2^-11)
    errs = {"logits": rel_err(logits, want), "h": rel_err(g.Peek("h", E), cpu.last_h()),
            "up": rel_err(g.Peek("up", (row + 1) * F)[row * F:], cpu.last_up()),
            "k": rel_err(g.Peek("k", kvd), cpu.kv_row(L - 1, n - 1)),
            "v": rel_err(g.Peek("v", kvd), cpu.kv_row(L - 1, n - 1, v=True))}
    print(f"{name} {n}: " + " ".join(f"{k} {v:.2e}" for k, v in errs.items()), flush=True)
    assert errs.pop("logits") <= LOGIT_TOL and max(errs.values()) <= tol
    toks, lgs = cpu_greedy(cpu, prompt, 6)
    greedy_parity(g, prompt, toks, lgs)


def test_wide_and_chunked_agree(gpu):
    """A budget too small for the wide buffers leaves the chunked prefill:
    the same calls, results within f32 rounding of each other; Layers and its
    trace read the same rows."""
    from llm_amd import llm
    spec = synth.tiny_qwen(seed=45, layers=3, ctx=2048)
    path = synth.cached(spec)
    g = llm.NewGPU(0, None, path, 1152)
    lim = llm.DefaultLimits()
    lim.memory_budget = g.MemoryUsed() - 1
    c = llm.NewGPU(0, lim, path, 1152)
    assert c.MemoryUsed() < g.MemoryUsed()
    prompt = [int(t) for t in synth.prompt(46, 200, spec.vocab)]
    rows = (len(prompt) - 1) % 64 + 1
    for layers in (0, 1, 2):
        g.Layers = c.Layers = layers
        lg, lc = g.PrefillLogits(prompt), c.PrefillLogits(prompt)
        for name, w in (("x", spec.embd), ("q", spec.embd), ("att", spec.embd), ("gate", spec.ff), ("up", spec.ff)):
            assert rel_err(g.Peek(name, rows * w), c.Peek(name, rows * w)) <= 1e-5, (layers, name)
        if layers == 0:
            assert rel_err(lg, lc) <= 1e-5
            assert gpu_generate(g, prompt, 12) == gpu_generate(c, prompt, 12)
    assert np.array_equal(g.Peek("tokens", len(prompt)), c.Peek("tokens", len(prompt)))
