"""The decode step of one to four sequences in one launch (ternaspmm_decode_step) against the launches it stands for: the same
bits in the logits and in the caches, whatever the shape, the prefix, the quantisation mode or the values."""
import ctypes

import pytest
import torch

from ternainfer_amd import _lib
from ternainfer_amd.model import ModelArgs, Transformer, greedy_decode

pytestmark = pytest.mark.gpu

# heads, kv heads, ffn: one head a group and several, K of one tile run and of a remainder of one, the widest
TINY, ODD, WIDE = dict(n_heads=2, n_kv_heads=1, ffn_dim=192), dict(n_heads=9, n_kv_heads=3, ffn_dim=1088), dict(n_heads=20, n_kv_heads=5, ffn_dim=6912)
WIDEST = dict(n_heads=20, n_kv_heads=5, ffn_dim=7168)
SINGLE = dict(n_heads=5, n_kv_heads=5, ffn_dim=64)


def build(shape, layers, seed=3):
    args = ModelArgs(dim=128 * shape["n_heads"], n_layers=layers, vocab_size=512, **shape)
    model = Transformer(args, seed=seed)
    for i, blk in enumerate(model.layers):            # norm weights that are not all one
        gen = torch.Generator(device="cuda").manual_seed(100 + i)
        for name in ("attention_norm", "attn_sub_norm", "ffn_norm", "ffn_sub_norm"):
            w = getattr(blk, name)
            w.copy_(torch.randn(w.shape, generator=gen, device="cuda").mul_(0.3).add_(1.0))
    return model


def state(model, m, slots, positions, seed=5):
    a = model.args
    gen = torch.Generator(device="cuda").manual_seed(seed)
    whole = torch.randn((a.n_layers, 2, m, a.n_kv_heads, slots, a.head_dim), generator=gen, device="cuda").to(torch.bfloat16)
    tokens = torch.randint(0, a.vocab_size, (m, 1), generator=gen, device="cuda")
    pos = torch.tensor([[p] for p in positions] if len(positions) > 1 or m == 1 else positions, dtype=torch.int64, device="cuda")
    return whole, tokens, pos


def step(model, whole, tokens, pos, one_launch):
    """(logits, caches) of a step; asserts that the launch takes it, or leaves it to the launches it stands for."""
    held = whole.clone()
    cache = [(held[i, 0], held[i, 1]) for i in range(model.args.n_layers)]
    model.one_launch_step = one_launch
    with torch.inference_mode():
        if one_launch:
            assert model.whole_step(tokens, cache, pos, whole.shape[4]) is not None
            held.copy_(whole)
            return model.forward(tokens, cache, pos), held
        model.defer_above = 8192                      # the launches with the attention in one piece
        try:
            return model.forward(tokens, cache, pos), held
        finally:
            del model.defer_above


def same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def check(model, whole, tokens, pos):
    want, want_cache = step(model, whole, tokens, pos, False)
    got, got_cache = step(model, whole, tokens, pos, True)
    assert same(got, want) and same(got_cache, want_cache)
    return got


@pytest.mark.parametrize("shape,m,slots,positions", [
    (TINY, 1, 64, [0]), (TINY, 1, 65, [64]), (TINY, 2, 1, [0]), (TINY, 4, 17, [16, 0, 15, 7]), (SINGLE, 1, 128, [127]), (SINGLE, 3, 40, [39]),
    (ODD, 1, 200, [130]), (ODD, 2, 640, [639, 513]), (ODD, 3, 129, [128]), (ODD, 4, 640, [1, 639, 127, 128]), (ODD, 1, 1030, [1029]), (ODD, 1, 8192, [8191]),
    (WIDE, 1, 384, [255]), (WIDE, 1, 1024, [1023]), (WIDE, 2, 101, [100]), (WIDE, 3, 101, [100, 50, 0]), (WIDE, 4, 640, [639]), (WIDE, 4, 1024, [1023, 640, 0, 777]), (WIDE, 2, 1280, [1279, 1024]), (ODD, 3, 1001, [1000]), (WIDEST, 1, 300, [16]), (WIDEST, 4, 100, [99]),
])
def test_one_launch_gives_the_bits_of_the_launches(shape, m, slots, positions):
    model = build(shape, 3)
    logits = check(model, *state(model, m, slots, positions))
    assert torch.isfinite(logits.float()).all()


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("m", [1, 2, 4])
def test_quantisation_modes(mode, m):
    """One sequence in every mode; more not in the eager one, whose integers fill the byte: there the launches run."""
    lib = _lib.load()
    model = build(ODD, 2)
    s = state(model, m, 100, [77])
    before = lib.ternaspmm_quant_mode(mode)
    try:
        if mode == 2 and m > 1:
            whole, tokens, pos = s
            with torch.inference_mode():
                assert model.whole_step(tokens, [(whole[i, 0], whole[i, 1]) for i in range(2)], pos, 100) is None
            assert torch.isfinite(model.forward(tokens, [(whole[i, 0], whole[i, 1]) for i in range(2)], pos).float()).all()
        else:
            check(model, *s)
    finally:
        lib.ternaspmm_quant_mode(before)


@pytest.mark.parametrize("m,positions", [(1, [-1]), (1, [500]), (3, [-7, 100, 1 << 40]), (2, [99, 99])])
def test_positions_outside_the_cache(m, positions):
    """Clamped, and no cache row is written for them -- as the launches do."""
    model = build(TINY, 2)
    check(model, *state(model, m, 100, positions))


@pytest.mark.parametrize("m", [1, 3])
def test_rows_that_are_not_finite(m):
    """A NaN of any payload, also the two that stand for a word that has not come, and an infinity in a row's embedding: its
    logits are NaN, the other rows are untouched."""
    model = build(ODD, 2)
    for bits in (0x7fc0, 0xffff, 0x7f80):
        whole, tokens, pos = state(model, m, 100, [60])
        model.tok_embeddings[7, 4:6] = torch.tensor([bits, bits], dtype=torch.int32, device="cuda").to(torch.int16).view(torch.bfloat16)
        tokens[0] = 7
        tokens[1:] = 9
        want, _ = step(model, whole, tokens, pos, False)
        got, _ = step(model, whole, tokens, pos, True)
        assert torch.isnan(got[0].float()).all() and torch.isnan(want[0].float()).all()
        assert same(got[1:], want[1:]) and torch.isfinite(got[1:, :7].float()).all()


def test_a_switch_of_one_block_asks_for_the_launches():
    """As one of the model, or of all blocks, does: whoever sets it times or checks the launches."""
    from ternainfer_amd.model import _CHAIN_SWITCHES, Block
    model = build(TINY, 3)
    whole, tokens, pos = state(model, 2, 40, [11])
    cache = [(whole[i, 0], whole[i, 1]) for i in range(3)]
    with torch.inference_mode():
        for name, default in _CHAIN_SWITCHES:
            assert getattr(Block, name) == default
            setattr(model.layers[1], name, (not default) if isinstance(default, bool) else default - 1)
            assert model.whole_step(tokens, cache, pos, 40) is None, name
            assert torch.isfinite(model.forward(tokens, cache, pos).float()).all()
            delattr(model.layers[1], name)
            assert model.whole_step(tokens, cache, pos, 40) is not None, name


def test_more_blocks_than_a_launch_takes():
    model = build(TINY, 65)
    check(model, *state(model, 1, 64, [33]))
    check(model, *state(model, 3, 30, [29, 2, 11]))


def test_greedy_tokens_are_those_of_the_launches():
    model = build(ODD, 4)
    prompt = torch.randint(0, 512, (3, 19), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    tokens = {}
    for on in (False, True):
        model.one_launch_step = on
        tokens[on] = greedy_decode(model, prompt, 12)[0]
    assert torch.equal(tokens[False], tokens[True])


def test_steps_on_several_streams_at_once():
    """Four captured steps replayed on four streams side by side: their grids wait within themselves only."""
    model = build(WIDE, 4)
    runs = []
    for i, m in enumerate((1, 3, 1, 2)):
        whole, tokens, pos = state(model, m, 120, [100], seed=20 + i)
        want, _ = step(model, whole, tokens, pos, False)
        cache = [(whole[n, 0], whole[n, 1]) for n in range(4)]
        model.one_launch_step = True
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.inference_mode():
            with torch.cuda.stream(stream):
                model.forward(tokens, cache, pos)
            torch.cuda.current_stream().wait_stream(stream)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                logits = model.forward(tokens, cache, pos)
        runs.append((stream, graph, logits, want, cache, tokens, pos))
    torch.cuda.synchronize()
    for _ in range(3):
        for _ in range(8):
            for stream, graph, *_ in runs:
                with torch.cuda.stream(stream):
                    graph.replay()
        torch.cuda.synchronize()
        with torch.inference_mode():
            for _, _, logits, want, *_ in runs:
                assert same(logits, want)
                logits.zero_()
        torch.cuda.synchronize()


def test_split_attention_steps_of_two_streams_at_once():
    """Two captured steps of one model and one batch size whose launches leave partial attention results, side by side: each has
    its own."""
    model = build(WIDE, 4)
    runs = []
    for i in range(2):
        whole, tokens, pos = state(model, 6, 700, [690 - 30 * i], seed=40 + i)
        assert model.attention_partial(6, 700)[1] > 1 and model.whole_step(tokens, [(whole[n, 0], whole[n, 1]) for n in range(4)], pos, 700) is None
        cache = [(whole[n, 0], whole[n, 1]) for n in range(4)]
        stream = torch.cuda.Stream()
        with torch.inference_mode():
            want = model.forward(tokens, cache, pos).clone()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                logits = model.forward(tokens, cache, pos)
        runs.append((stream, graph, logits, want, cache, tokens, pos))
    torch.cuda.synchronize()
    for _ in range(3):
        for _ in range(8):
            for stream, graph, *_ in runs:
                with torch.cuda.stream(stream):
                    graph.replay()
        torch.cuda.synchronize()
        for _, _, logits, want, *_ in runs:
            assert same(logits, want)


class StepBlock(ctypes.Structure):
    """ternaspmm_step_block of include/ternaspmm.h."""
    _fields_ = [(n, ctypes.c_void_p) for n in ("wqkv", "wo", "w13", "w2", "ws_qkv", "ws_o", "ws_13", "ws_down", "attention_norm", "attn_sub_norm", "ffn_norm",
                                               "ffn_sub_norm", "cache_k", "cache_v")]


class StepDesc(ctypes.Structure):
    """ternaspmm_step_desc of include/ternaspmm.h."""
    _fields_ = [(n, ctypes.c_int) for n in ("layers", "M", "dim", "ffn", "heads", "kv_heads", "head_dim", "slots", "splits", "per_sequence", "vocab",
                                            "ws_num_qkv", "ws_num_o", "ws_num_down")] + [("eps", ctypes.c_float), ("scale", ctypes.c_float)]


def raw_step(model, whole, tokens, pos, workgroups, polls):
    """(call, stream behind the last block): ternaspmm_probe_decode_step on the buffers of `state`; call() enqueues it."""
    a, lib = model.args, _lib.load()
    m, slots = whole.shape[2], whole.shape[4]
    b0 = model.layers[0]
    desc = StepDesc(a.n_layers, m, a.dim, a.ffn_dim, a.n_heads, a.n_kv_heads, a.head_dim, slots,
                    lib.ternaspmm_attention_partial_splits_kv(1, a.n_heads, a.n_kv_heads, slots) if m == 1 else 1, int(pos.numel() == m and m > 1), a.vocab_size,
                    b0.wqkv.ws_num, b0.wo.ws_num, b0.w2.ws_num, a.norm_eps, a.head_dim ** -0.5)
    blocks = (StepBlock * a.n_layers)(*[
        StepBlock(*(t.data_ptr() for t in (b.wqkv.packed, b.wo.packed, b.gate_up_interleaved(), b.w2.packed, b.wqkv.ws, b.wo.ws, b.w13.ws, b.w2.ws, b.attention_norm,
                                           b.attn_sub_norm, b.ffn_norm, b.ffn_sub_norm, whole[i, 0], whole[i, 1]))) for i, b in enumerate(model.layers)])
    table = model.rope_tables(slots, whole.device)
    scratch = torch.empty(lib.ternaspmm_decode_step_bytes(ctypes.byref(desc)), dtype=torch.uint8, device="cuda")
    x = torch.zeros((m, a.dim), dtype=torch.bfloat16, device="cuda")
    held = (blocks, table, scratch, tokens, pos)

    def call():
        assert held and lib.ternaspmm_probe_decode_step(
            ctypes.byref(desc), blocks, tokens.data_ptr(), pos.data_ptr(), model.tok_embeddings.data_ptr(), table.data_ptr(), scratch.data_ptr(), x.data_ptr(),
            workgroups, polls, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    return call, x


@pytest.mark.parametrize("shape,layers,m,slots,positions,workgroups,polls", [
    (TINY, 3, 1, 64, [40], 1, 1), (TINY, 65, 1, 64, [33], 255, 512), (TINY, 65, 3, 30, [29, 2, 11], 16, 1), (SINGLE, 2, 2, 128, [127], 255, 1),
    (ODD, 3, 1, 200, [130], 100, 256), (ODD, 3, 4, 640, [1, 639, 127, 128], 200, 1), (ODD, 2, 1, 8192, [8191], 64, 1),
    (WIDE, 2, 1, 384, [255], 240, 1024), (WIDE, 2, 2, 101, [100], 255, 1), (WIDE, 2, 4, 1024, [1023, 640, 0, 777], 128, 1), (WIDE, 2, 1, 384, [300], 256, 1),
])
def test_a_step_whose_workgroups_do_not_all_come(shape, layers, m, slots, positions, workgroups, polls):
    """Fewer workgroups than wait for each other, and waits that end soon: the step is done again in order, with the same bits in
    the stream and in the caches -- eager, captured, and after a step that went through."""
    model = build(shape, layers)
    whole, tokens, pos = state(model, m, slots, positions)
    fresh = whole.clone()
    call, x = raw_step(model, whole, tokens, pos, 256, 131072)
    call()
    want, want_cache = x.clone(), whole.clone()
    assert torch.isfinite(want.float()).all()
    whole.copy_(fresh)
    short, x = raw_step(model, whole, tokens, pos, workgroups, polls)
    short()
    assert same(x, want) and same(whole, want_cache)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        short()
    for _ in range(3):
        whole.copy_(fresh)
        x.fill_(7.0)
        graph.replay()
        assert same(x, want) and same(whole, want_cache)
