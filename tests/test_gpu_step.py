"""GPU parity of the whole decode step (LiteSparkQwen.forward_token,
cpu_lightspark.py:424-468 in the reference repository) against the CPU
oracle: logits, KV cache and greedy tokens bit-exact."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import assert_bits_equal, assert_bits_or_nan_equal, dev, to_dev, to_host

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

KEYS = ("qkv", "qkv_scales", "o", "o_scales", "gate_up", "gate_up_scales", "down",
        "down_scales", "input_norm", "post_norm", "q_norm", "k_norm")


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu] {request.node.nodeid}", flush=True)
    yield
    torch.cuda.synchronize()


def golden_model(g):
    from harsh4b_amd.synthetic import model_from_arrays
    arrays = {k: [np.ascontiguousarray(a) for a in g[k]] for k in KEYS}
    for k in ("embedding", "embedding_scales", "final_norm"):
        arrays[k] = np.ascontiguousarray(g[k])
    return model_from_arrays(g["config"], arrays)


def oracle_of(model):
    from harsh4b_amd.synthetic import host_arrays
    return oracle.OracleModel(model.config, host_arrays(model))


def test_rope_tables_match_reference_run(forward_golden):
    from harsh4b_amd.lightspark import rope_tables
    cos, sin = rope_tables(forward_golden["config"])
    np.testing.assert_array_equal(cos, forward_golden["rope_cos"])
    np.testing.assert_array_equal(sin, forward_golden["rope_sin"])


def test_tiny_model_step_by_step(forward_golden):
    g = forward_golden
    model = golden_model(g)
    ref = oracle_of(model)
    cap = len(g["tokens"])
    st = model.new_state(cap)
    rs = ref.new_state(cap)
    for i, t in enumerate(g["tokens"]):
        logits = model.forward_token(int(t), st)
        tok = model.greedy_token(st)
        rtok = ref.forward_token(int(t), rs)
        assert_bits_equal(to_host(logits), rs.logits, f"logits step {i}")
        assert tok == rtok == int(g["greedy"][i]), (i, tok, rtok, g["greedy"][i])
        # the reference run used an fp32 KV cache: fp16 storage stays close
        assert np.abs(to_host(logits) - g["logits"][i]).max() < 0.1
    assert_bits_equal(to_host(st.keys).view(np.uint16), rs.keys, "keys")
    assert_bits_equal(to_host(st.values).view(np.uint16), rs.values, "values")
    assert_bits_equal(to_host(st.x), rs.x, "residual")
    st.check_status()


def test_tiny_model_graph_replay_matches_eager(forward_golden):
    g = forward_golden
    model = golden_model(g)
    a = model.new_state(12)
    b = model.new_state(12)
    first = int(g["tokens"][0])
    # eager greedy loop
    toks_a = []
    model.forward_token(first, a)
    for _ in range(8):
        t = model.greedy_token(a)
        toks_a.append(t)
        model.forward_token(t, a)
    toks_a.append(model.greedy_token(a))
    # device-resident greedy loop through a captured graph, replayed 9 times
    toks_b = []
    with torch.cuda.stream(b.stream):
        b.token.fill_(first)
    for _ in range(9):
        model.decode_greedy(b, 1)
        toks_b.append(model.greedy_token(b))
    assert toks_a == toks_b
    assert_bits_equal(to_host(b.logits), to_host(a.logits), "graph logits")
    assert_bits_equal(to_host(b.keys).view(np.uint16), to_host(a.keys).view(np.uint16), "graph keys")
    a.check_status()
    b.check_status()


def test_step_errors(forward_golden):
    g = forward_golden
    model = golden_model(g)
    st = model.new_state(1)
    with pytest.raises(ValueError, match="outside the vocabulary"):
        model.forward_token(int(g["config"]["vocab_size"]), st)
    model.forward_token(3, st)
    with pytest.raises(ValueError, match="capacity exhausted"):
        model.forward_token(3, st)


def test_device_flags_bad_token_without_fault(forward_golden):
    # force the condition from the host: an out-of-vocabulary id written
    # straight into the device token slot; the kernel clamps and flags it
    import ctypes
    from harsh4b_amd import _native
    g = forward_golden
    model = golden_model(g)
    st = model.new_state(2)
    with torch.cuda.stream(st.stream):
        st.token.fill_(10 ** 6)
    _native.check(_native.lib().hq_decode_step(ctypes.byref(model.struct), ctypes.byref(st.struct),
                                               st.stream.cuda_stream), "step")
    with pytest.raises(ValueError, match="outside the vocabulary"):
        st.check_status()


# ------------------------------------------------------------------ full size
@pytest.fixture(scope="module")
def qwen():
    from harsh4b_amd.config import QWEN3_4B
    from harsh4b_amd.synthetic import random_model
    model = random_model(QWEN3_4B, seed=11)
    torch.cuda.synchronize()
    return model, oracle_of(model)


def test_qwen3_4b_first_tokens_bit_exact(qwen):
    model, ref = qwen
    cap = 8
    st = model.new_state(cap)
    rs = ref.new_state(cap)
    token = 151643
    for i in range(4):
        logits = model.forward_token(token, st)
        tok = model.greedy_token(st)
        rtok = ref.forward_token(token, rs)
        assert_bits_equal(to_host(logits), rs.logits, f"logits step {i}")
        assert tok == rtok
        token = tok
    assert_bits_equal(to_host(st.keys).view(np.uint16)[:, :4], rs.keys[:, :4], "keys")
    st.check_status()


@pytest.mark.parametrize("ctx", [100, 130, 300, 4000, 4096, 4097])
def test_qwen3_4b_long_context_bit_exact(qwen, ctx):
    # an fp16 N(0,1) cache of `ctx` positions on both sides, then two steps.
    # ctx 4000: 63-chunk contexts; 4096 and 4097: 65 and 66 chunks of 64
    # positions, more attention items than one round of blocks
    model, ref = qwen
    cap = ctx + 2
    st = model.new_state(cap)
    rs = ref.new_state(cap)
    rng = np.random.default_rng(ctx)
    shape = st.keys.shape
    for name in ("keys", "values"):
        cache = rng.standard_normal((shape[0], ctx) + tuple(shape[2:])).astype(np.float16)
        getattr(st, name)[:, :ctx] = to_dev(cache)
        getattr(rs, name)[:, :ctx] = cache.view(np.uint16)
    st.device_position.fill_(ctx)
    st.position = ctx
    rs.position = ctx
    torch.cuda.synchronize()
    token = 1234
    for i in range(2):
        logits = model.forward_token(token, st)
        tok = model.greedy_token(st)
        rtok = ref.forward_token(token, rs)
        assert_bits_equal(to_host(logits), rs.logits, f"ctx {ctx} step {i}")
        assert tok == rtok
        token = tok
    assert_bits_equal(to_host(st.keys).view(np.uint16)[:, ctx:ctx + 2], rs.keys[:, ctx:ctx + 2], "new keys")
    st.check_status()


# ------------------------------------------- persistent layer kernel vs per-layer
def _run_tokens(model, st, tokens):
    out = []
    for t in tokens:
        out.append(to_host(model.forward_token(int(t), st)).copy())
    return out


def test_tiny_model_layer_kernel_matches_per_layer_kernels(forward_golden):
    g = forward_golden
    model = golden_model(g)
    assert model.layer_kernel_blocks > 0, "the tiny model fits the persistent layer kernel"
    cap = len(g["tokens"])
    a = model.new_state(cap)
    la = _run_tokens(model, a, g["tokens"])
    model.per_layer_kernels = True
    assert model.layer_kernel_blocks == 0
    b = model.new_state(cap)
    lb = _run_tokens(model, b, g["tokens"])
    model.per_layer_kernels = False
    for i, (x, y) in enumerate(zip(la, lb)):
        assert_bits_equal(x, y, f"logits step {i}")
    assert_bits_equal(to_host(a.keys).view(np.uint16), to_host(b.keys).view(np.uint16), "keys")
    assert_bits_equal(to_host(a.x), to_host(b.x), "residual")
    a.check_status()
    b.check_status()


@pytest.mark.parametrize("ctx", [0, 200, 300])
def test_qwen3_4b_layer_kernel_matches_per_layer_kernels(qwen, ctx):
    model, _ = qwen
    assert model.layer_kernel_blocks > 0, "Qwen3-4B fits the persistent layer kernel"
    cap = ctx + 4
    states = []
    rng = np.random.default_rng(ctx + 7)
    cache = {}
    for name in ("keys", "values"):
        cache[name] = rng.standard_normal((36, ctx, 8, 128)).astype(np.float16)
    results = []
    for per_layer in (False, True):
        model.per_layer_kernels = per_layer
        st = model.new_state(cap)
        if ctx:
            for name in ("keys", "values"):
                getattr(st, name)[:, :ctx] = to_dev(cache[name])
            st.device_position.fill_(ctx)
            st.position = ctx
            torch.cuda.synchronize()
        toks, logits = [], []
        token = 4242
        for _ in range(3):
            logits.append(to_host(model.forward_token(token, st)).copy())
            token = model.greedy_token(st)
            toks.append(token)
        st.check_status()
        results.append((toks, logits, to_host(st.keys).view(np.uint16)[:, ctx:ctx + 3].copy()))
        states.append(st)
    model.per_layer_kernels = False
    (ta, la, ka), (tb, lb, kb) = results
    assert ta == tb
    for i in range(3):
        assert_bits_equal(la[i], lb[i], f"ctx {ctx} logits step {i}")
    assert_bits_equal(ka, kb, f"ctx {ctx} new keys")


def test_layer_kernel_graph_replays_continue_epochs(forward_golden):
    # the hand-off epochs live in the workspace: many replays of one captured
    # step stay in step with eager steps of the per-layer path
    g = forward_golden
    model = golden_model(g)
    first = int(g["tokens"][0])
    a = model.new_state(40)
    with torch.cuda.stream(a.stream):
        a.token.fill_(first)
    toks_a = []
    for _ in range(30):
        model.decode_greedy(a, 1)
        toks_a.append(model.greedy_token(a))
    model.per_layer_kernels = True
    b = model.new_state(40)
    toks_b = []
    model.forward_token(first, b)
    for _ in range(29):
        t = model.greedy_token(b)
        toks_b.append(t)
        model.forward_token(t, b)
    toks_b.append(model.greedy_token(b))
    model.per_layer_kernels = False
    assert toks_a == toks_b
    assert_bits_equal(to_host(a.logits), to_host(b.logits), "logits after 30 steps")
    a.check_status()
    b.check_status()


class SamplerArgs:
    argmax = False

    def __init__(self, temperature=0.7, top_k=40, top_p=0.9, repetition_penalty=1.08):
        self.temperature, self.top_k, self.top_p = temperature, top_k, top_p
        self.repetition_penalty = repetition_penalty


def test_tiny_model_sampled_decode_matches_oracle(forward_golden):
    # the reference's stochastic loop (cpu_lightspark.py:808-880): sample
    # after the prompt with nothing generated, then append, forward, sample
    from harsh4b_amd.lightspark import sample_logits
    g = forward_golden
    model = golden_model(g)
    ref = oracle_of(model)
    args = SamplerArgs(temperature=1.0, top_k=12, top_p=0.95, repetition_penalty=1.3)
    prompt = [int(t) for t in g["tokens"][:4]]
    steps = 10
    st, rs = model.new_state(len(prompt) + steps), ref.new_state(len(prompt) + steps)
    g_dev, g_ref = np.random.default_rng(9), np.random.default_rng(9)
    for t in prompt:
        logits = model.forward_token(t, st)
        ref.forward_token(t, rs)
    first = sample_logits(logits, [], args, g_dev)
    want = [oracle.sample_token(rs.logits, [], 1.3, 1.0, 12, 0.95, g_ref.random())[0]]
    assert first == want[0]
    for _ in range(steps):
        ref.forward_token(want[-1], rs)
        want.append(oracle.sample_token(rs.logits, want, 1.3, 1.0, 12, 0.95, g_ref.random())[0])
    got = [first] + model.decode_sampled(st, steps, args, g_dev, [first])
    assert got == want
    assert_bits_equal(to_host(st.logits), rs.logits, "logits after the loop")
    assert g_dev.random() == g_ref.random()
    st.check_status()


def test_qwen3_4b_sampled_decode_matches_per_op_sampler(qwen):
    # the device loop against forward_token + sample_logits per token, with
    # the reference runner's default policy
    from harsh4b_amd.lightspark import sample_logits
    model, _ = qwen
    args = SamplerArgs()
    steps = 8
    a, b = model.new_state(steps + 2), model.new_state(steps + 2)
    g_a, g_b = np.random.default_rng(0), np.random.default_rng(0)
    generated = [4242]
    for _ in range(steps):
        generated.append(sample_logits(model.forward_token(generated[-1], a), generated, args, g_a))
    got = model.decode_sampled(b, steps, args, g_b, [4242])
    assert got == generated[1:]
    assert_bits_equal(to_host(a.logits), to_host(b.logits), "logits")
    a.check_status()
    b.check_status()


def _prefill_vs_steps(model, prompt, cap, start_tokens=()):
    """Batched prefill against forward_token per token: K/V rows, logits,
    greedy token and position, bit for bit."""
    a, b = model.new_state(cap), model.new_state(cap)
    for t in start_tokens:                       # an earlier turn, decoded token by token
        model.forward_token(int(t), a)
        model.forward_token(int(t), b)
    la = to_host(model.prefill(prompt, a)).copy()
    for t in prompt:
        lb = model.forward_token(int(t), b)
    lb = to_host(lb).copy()
    n = len(start_tokens) + len(prompt)
    assert a.position == b.position == n
    assert int(a.device_position.item()) == n
    assert_bits_equal(to_host(a.keys)[:, :n].view(np.uint16), to_host(b.keys)[:, :n].view(np.uint16), "keys")
    assert_bits_equal(to_host(a.values)[:, :n].view(np.uint16), to_host(b.values)[:, :n].view(np.uint16),
                      "values")
    assert_bits_equal(la, lb, "logits after the prompt")
    assert model.greedy_token(a) == model.greedy_token(b)
    a.check_status()
    b.check_status()
    return a


@pytest.mark.parametrize("n", [1, 2, 5, 10])
def test_tiny_model_prefill_matches_token_steps(forward_golden, n):
    g = forward_golden
    model = golden_model(g)
    prompt = [int(t) for t in g["tokens"][:n]]
    st = _prefill_vs_steps(model, prompt, 16)
    # and against the oracle
    ref = oracle_of(model)
    rs = ref.new_state(16)
    for t in prompt:
        ref.forward_token(t, rs)
    assert_bits_equal(to_host(st.logits), rs.logits, "oracle logits")
    _prefill_vs_steps(model, prompt, 24, start_tokens=[3, 4, 5])


def test_tiny_model_prefill_flags_bad_tokens(forward_golden):
    g = forward_golden
    model = golden_model(g)
    st = model.new_state(8)
    with pytest.raises(ValueError, match="outside the vocabulary"):
        model.prefill([1, int(g["config"]["vocab_size"])], st)
    with pytest.raises(ValueError, match="capacity"):
        model.prefill(list(range(9)), st)
    assert st.position == 0


def test_qwen3_4b_prefill_matches_token_steps(qwen):
    # 200 tokens after two: contexts of up to four chunks, the layer kernel for
    # the comparison steps
    model, _ = qwen
    rng = np.random.default_rng(21)
    prompt = [int(t) for t in rng.integers(0, 151936, 200)]
    _prefill_vs_steps(model, prompt, 208, start_tokens=[11, 12])


def test_qwen3_4b_prefill_after_a_long_turn(qwen):
    # a 300-token prompt after a 300-token earlier turn: query contexts 301-600
    # (up to ten chunks)
    model, _ = qwen
    rng = np.random.default_rng(33)
    earlier = [int(t) for t in rng.integers(0, 151936, 300)]
    prompt = [int(t) for t in rng.integers(0, 151936, 300)]
    _prefill_vs_steps(model, prompt, 604, start_tokens=earlier)


@pytest.mark.parametrize("start,n", [(0, 66), (1, 15), (63, 2), (60, 150), (511, 17), (1000, 130), (0, 1050)])
def test_qwen3_4b_prefill_attention_forms(qwen, start, n):
    # query tiles aligned to 16 positions that begin and end inside one, on
    # both sides of a 64-position chunk edge: single-chunk batches, chunk
    # partials with their combine, and (1050 tokens) the stored scores
    model, _ = qwen
    rng = np.random.default_rng(7 * start + n)
    a, b = model.new_state(start + n), model.new_state(start + n)
    if start:
        earlier = [int(t) for t in rng.integers(0, 151936, start)]
        model.prefill(earlier, a)
        for t in earlier:
            model.forward_token(t, b)
    prompt = [int(t) for t in rng.integers(0, 151936, n)]
    la = to_host(model.prefill(prompt, a)).copy()
    for t in prompt:
        lb = model.forward_token(t, b)
    assert_bits_equal(to_host(a.keys).view(np.uint16), to_host(b.keys).view(np.uint16), "keys")
    assert_bits_equal(to_host(a.values).view(np.uint16), to_host(b.values).view(np.uint16), "values")
    assert_bits_equal(la, to_host(lb), "logits")
    a.check_status()
    b.check_status()


@pytest.mark.parametrize("heads,kv", [(16, 8), (6, 2), (3, 3), (8, 2)])
def test_prefill_attention_mixed_blocks(heads, kv):
    # head counts and starts for which a block's four (tile, head) slots mix
    # tiles of one chunk and of two (never with four heads per kv head)
    from harsh4b_amd.synthetic import random_model
    config = {"hidden_size": 256, "intermediate_size": 512, "num_attention_heads": heads, "num_key_value_heads": kv,
              "head_dim": 128, "num_hidden_layers": 2, "vocab_size": 515, "rms_norm_eps": 1e-6,
              "rope_theta": 1000000, "max_position_embeddings": 1024}
    model = random_model(config, 5, dev())
    rng = np.random.default_rng(heads)
    for start in (16, 20, 33, 48, 60):
        earlier = [int(t) for t in rng.integers(0, 515, start)]
        for n in (45, 60, 300):
            _prefill_vs_steps(model, [int(t) for t in rng.integers(0, 515, n)], start + n, start_tokens=earlier)


@pytest.mark.parametrize("heads,kv", [(16, 8), (8, 2), (2, 2)])
@pytest.mark.parametrize("start", [61, 62, 64, 700, 4158])
def test_prefill_of_few_queries(heads, kv, start):
    # one and two queries (a block per query, head and chunk) and three (tiles
    # of 16), their contexts on both sides of a chunk edge
    from harsh4b_amd.synthetic import random_model
    config = {"hidden_size": 256, "intermediate_size": 512, "num_attention_heads": heads, "num_key_value_heads": kv,
              "head_dim": 128, "num_hidden_layers": 2, "vocab_size": 515, "rms_norm_eps": 1e-6,
              "rope_theta": 1000000, "max_position_embeddings": 8192}
    model = random_model(config, 6, dev())
    rng = np.random.default_rng(start)
    for n in (2, 3, 4):                          # the last token goes through the decode step
        prompt = [int(t) for t in rng.integers(0, 515, n)]
        a, b = model.new_state(start + n), model.new_state(start + n)
        for cache in ("keys", "values"):
            hist = torch.randn((2, start, kv, 128), generator=torch.Generator(dev()).manual_seed(n), device=dev()).half()
            getattr(a, cache)[:, :start] = hist
            getattr(b, cache)[:, :start] = hist
        a.device_position.fill_(start)
        b.device_position.fill_(start)
        model.stream.wait_stream(torch.cuda.current_stream())
        a.position = b.position = start
        la = to_host(model.prefill(prompt, a)).copy()
        for t in prompt:
            lb = model.forward_token(t, b)
        assert_bits_equal(to_host(a.keys).view(np.uint16), to_host(b.keys).view(np.uint16), f"{n} keys")
        assert_bits_equal(to_host(a.values).view(np.uint16), to_host(b.values).view(np.uint16), f"{n} values")
        assert_bits_equal(la, to_host(lb), f"{n} logits")
        a.check_status()
        b.check_status()


@pytest.mark.parametrize("heads,kv,start,n", [(16, 8, 20, 100), (16, 8, 200, 3), (8, 2, 200, 150), (16, 8, 200, 1100),
                                              (3, 3, 130, 40)])
def test_prefill_attention_infinities_and_nan(heads, kv, start, n):
    # cache rows past the prompt hold infinities and NaN; then keys of huge
    # values, and in the second of three layers values of +-inf and NaN and an
    # infinite key: chunk partials and (1100 tokens) stored scores against
    # pieces of two tokens, which take one query per block
    import ctypes

    from harsh4b_amd import _native
    from harsh4b_amd.synthetic import random_model
    config = {"hidden_size": 256, "intermediate_size": 512, "num_attention_heads": heads, "num_key_value_heads": kv,
              "head_dim": 128, "num_hidden_layers": 3, "vocab_size": 515, "rms_norm_eps": 1e-6,
              "rope_theta": 1000000, "max_position_embeddings": 2048}
    model = random_model(config, 7, dev())
    lib = _native.lib()
    rng = np.random.default_rng(start + n)
    ids = to_dev(rng.integers(0, 515, n).astype(np.int32))
    ws = torch.empty(lib.hq_prefill_workspace_bytes(ctypes.byref(model.struct), start + n), dtype=torch.uint8,
                     device=dev())
    for infinite in (False, True):
        states = [model.new_state(start + n + 80) for _ in range(2)]
        for st in states:
            for cache in (st.keys, st.values):
                gen = torch.Generator(device=dev()).manual_seed(9)
                cache[:, :start] = torch.randn((3, start, kv, 128), generator=gen, device=dev()).half()
            st.keys[:, start // 2, 0, 7] = 60000.0
            st.keys[:, start - 1, kv - 1, 100] = -60000.0
            if infinite:
                st.values[1, start // 3, 0, 5] = float("inf")
                st.values[1, start - 2, kv - 1, 0] = float("-inf")
                st.values[1, 0, 0, 1] = float("nan")
                st.keys[1, 1, 0, 3] = float("inf")
            st.keys[:, start + n:] = float("inf")
            st.values[:, start + n:] = float("nan")
        torch.cuda.synchronize()
        for st, piece in zip(states, (n, 2)):
            for i in range(0, n, piece):
                assert lib.hq_prefill(ctypes.byref(model.struct), ctypes.byref(st.struct), ids[i:].data_ptr(),
                                      min(piece, n - i), start + i, ws.data_ptr(), model.stream.cuda_stream) == 0
        for name in ("keys", "values"):
            x, y = (to_host(getattr(st, name))[:, :start + n].astype(np.float32) for st in states)
            assert_bits_or_nan_equal(x, y, f"{name} infinite={infinite}")
            assert infinite or np.isfinite(x).all()


@pytest.mark.parametrize("heads,kv,start,n", [(10, 2, 20, 150), (16, 2, 60, 300), (7, 1, 37, 64), (12, 2, 0, 1500)])
def test_prefill_of_many_heads_per_kv_head(heads, kv, start, n):
    # five to eight query heads per kv head (the decode step takes up to four,
    # so the caches are the test's own): tiles against pieces of two tokens
    import ctypes

    from harsh4b_amd import _native
    from harsh4b_amd.synthetic import random_model
    config = {"hidden_size": 256, "intermediate_size": 512, "num_attention_heads": heads, "num_key_value_heads": kv,
              "head_dim": 128, "num_hidden_layers": 3, "vocab_size": 515, "rms_norm_eps": 1e-6,
              "rope_theta": 1000000, "max_position_embeddings": 2048}
    model = random_model(config, 10, dev())
    lib = _native.lib()
    rng = np.random.default_rng(n)
    ids = to_dev(rng.integers(0, 515, n).astype(np.int32))
    ws = torch.empty(lib.hq_prefill_workspace_bytes(ctypes.byref(model.struct), start + n), dtype=torch.uint8,
                     device=dev())
    caches = []
    for piece in (n, 2):
        gen = torch.Generator(device=dev()).manual_seed(11)
        keys, values = (torch.randn((3, start + n, kv, 128), generator=gen, device=dev()).half() for _ in range(2))
        position, status = (torch.zeros(1, dtype=torch.int32, device=dev()) for _ in range(2))
        st = _native.HqState()
        st.capacity = start + n
        st.keys, st.values = keys.data_ptr(), values.data_ptr()
        st.position, st.status = position.data_ptr(), status.data_ptr()
        torch.cuda.synchronize()
        for i in range(0, n, piece):
            assert lib.hq_prefill(ctypes.byref(model.struct), ctypes.byref(st), ids[i:].data_ptr(), min(piece, n - i),
                                  start + i, ws.data_ptr(), model.stream.cuda_stream) == 0
        torch.cuda.synchronize()
        assert int(position.item()) == start + n and int(status.item()) == 0
        caches.append((to_host(keys), to_host(values)))
    for x, y in zip(*caches):
        assert_bits_equal(x.view(np.uint16), y.view(np.uint16), f"{heads} / {kv}")


@pytest.mark.parametrize("heads,kv,start,n", [(16, 8, 5, 2060), (6, 2, 0, 4200), (32, 8, 201, 1100), (16, 8, 1000, 1300)])
def test_prefill_passes_and_stored_scores(heads, kv, start, n):
    # prompts of two and three passes of 2048 tokens, each with its own first
    # position, and stored scores of tiles that begin inside one past position 0
    from harsh4b_amd.synthetic import random_model
    config = {"hidden_size": 256, "intermediate_size": 512, "num_attention_heads": heads, "num_key_value_heads": kv,
              "head_dim": 128, "num_hidden_layers": 2, "vocab_size": 515, "rms_norm_eps": 1e-6,
              "rope_theta": 1000000, "max_position_embeddings": 8192}
    model = random_model(config, 8, dev())
    rng = np.random.default_rng(n)
    _prefill_vs_steps(model, [int(t) for t in rng.integers(0, 515, n)], start + n,
                      start_tokens=[int(t) for t in rng.integers(0, 515, start)])


def test_qwen3_4b_prefill_of_two_passes(qwen):
    # 2300 tokens in one call (2048 + 251) and in pieces within a pass
    model, _ = qwen
    rng = np.random.default_rng(2300)
    prompt = [int(t) for t in rng.integers(0, 151936, 2300)]
    a, b = model.new_state(2300), model.new_state(2300)
    la = to_host(model.prefill(prompt, a)).copy()
    for i in range(0, 2300, 900):
        lb = model.prefill(prompt[i:i + 900], b)
    assert_bits_equal(la, to_host(lb), "logits")
    assert_bits_equal(to_host(a.keys).view(np.uint16), to_host(b.keys).view(np.uint16), "keys")
    assert_bits_equal(to_host(a.values).view(np.uint16), to_host(b.values).view(np.uint16), "values")
    a.check_status()
    b.check_status()


def test_prefill_scratch_is_not_held_and_needs_no_clearing():
    # a prompt leaves no memory allocated with its state, gives the same bits
    # in a workspace of any contents, and stays within the bytes asked for
    import ctypes

    from harsh4b_amd import _native
    from harsh4b_amd.synthetic import random_model
    config = {"hidden_size": 352, "intermediate_size": 3232, "num_attention_heads": 6, "num_key_value_heads": 2,
              "head_dim": 128, "num_hidden_layers": 2, "vocab_size": 515, "rms_norm_eps": 1e-6,
              "rope_theta": 1000000, "max_position_embeddings": 1024}
    model = random_model(config, 4, dev())
    lib = _native.lib()
    side = torch.cuda.Stream()
    rng = np.random.default_rng(4)
    for n in (3, 20, 33, 65, 130, 600):
        prompt = [int(t) for t in rng.integers(0, 515, n)]
        a, b = model.new_state(700), model.new_state(700)
        torch.cuda.synchronize()
        held = torch.cuda.memory_allocated()
        with torch.cuda.stream(side):
            model.prefill(prompt, a)
            assert torch.cuda.memory_allocated() == held
            # what reuses the scratch's memory comes after the prompt
            reused = [torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=dev()) for nbytes in (1 << 20, 4 << 20, 8 << 20)]
        torch.cuda.synchronize()
        assert all(bool((r == 0xFF).all()) for r in reused)
        nbytes = lib.hq_prefill_workspace_bytes(ctypes.byref(model.struct), n - 1)
        ws = torch.full((nbytes + 65536,), 0xFF, dtype=torch.uint8, device=dev())   # (NaN as floats)
        ids = to_dev(np.array(prompt[:-1], np.int32))
        torch.cuda.synchronize()
        assert lib.hq_prefill(ctypes.byref(model.struct), ctypes.byref(b.struct), ids.data_ptr(), n - 1, 0,
                              ws.data_ptr(), model.stream.cuda_stream) == 0
        b.position = n - 1
        lb = to_host(model.forward_token(prompt[-1], b))
        assert bool((ws[nbytes:] == 0xFF).all())
        assert_bits_equal(to_host(a.logits), lb, f"{n} logits")
        assert_bits_equal(to_host(a.keys).view(np.uint16), to_host(b.keys).view(np.uint16), f"{n} keys")
        assert_bits_equal(to_host(a.values).view(np.uint16), to_host(b.values).view(np.uint16), f"{n} values")


def test_qwen3_4b_prefill_attention_scores_computed_twice(qwen):
    # 2000 tokens after 5000: the scores exceed the workspace, so the kernel
    # walks the keys twice; pieces of 300 tokens write chunk partials
    model, _ = qwen
    rng = np.random.default_rng(5)
    gen = torch.Generator(device=dev()).manual_seed(5)
    a, b = model.new_state(7000), model.new_state(7000)
    for cache in ("keys", "values"):
        hist = torch.randn((36, 5000, 8, 128), generator=gen, device=dev()).half()
        getattr(a, cache)[:, :5000] = hist
        getattr(b, cache)[:, :5000] = hist
    model.stream.wait_stream(torch.cuda.current_stream())
    a.position = b.position = 5000
    prompt = [int(t) for t in rng.integers(0, 151936, 2000)]
    la = to_host(model.prefill(prompt, a)).copy()
    for i in range(0, 2000, 300):
        lb = model.prefill(prompt[i:i + 300], b)
    assert_bits_equal(la, to_host(lb), "logits")
    assert_bits_equal(to_host(a.keys).view(np.uint16), to_host(b.keys).view(np.uint16), "keys")
    assert_bits_equal(to_host(a.values).view(np.uint16), to_host(b.values).view(np.uint16), "values")


@pytest.mark.parametrize("n", [33, 65, 130, 700])
def test_ragged_model_prefill_matches_token_steps(n):
    # widths that are no multiple of 128 columns, a row count of no tile:
    # the GEMMs in K parts, whole, and with SwiGLU in the epilogue
    from harsh4b_amd.synthetic import random_model
    config = {"hidden_size": 352, "intermediate_size": 3232, "num_attention_heads": 6, "num_key_value_heads": 2,
              "head_dim": 128, "num_hidden_layers": 3, "vocab_size": 515, "rms_norm_eps": 1e-6,
              "rope_theta": 1000000, "max_position_embeddings": 1024}
    model = random_model(config, 3, dev())
    rng = np.random.default_rng(n)
    _prefill_vs_steps(model, [int(t) for t in rng.integers(0, 515, n)], n + 8, start_tokens=[5, 6])
