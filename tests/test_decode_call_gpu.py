"""The ops' short incremental call and the general one give the same rows, the same step and the same errors."""
import pytest
import torch

from eet_amd import decoder as D
from eet_amd import ops


def decoders(alibi, rows):
    cfg = D.DecoderConfig(num_layers=1, hidden=256, heads=2, d_ff=704, vocab=64, alibi=alibi, max_batch=rows,
                          max_prompt=8, max_full_seq=12)
    sd, _ = D.random_state_dict(cfg, seed=5)
    return cfg, [D.Int8Decoder(cfg, sd, device="cuda:0").layers[0] for _ in range(2)]


@pytest.mark.gpu
@pytest.mark.parametrize("alibi", [False, True])
@pytest.mark.parametrize("rows", [1, 5, 32, 33])
def test_forms_of_one_call(gpu, alibi, rows):
    cfg, ((a, fa), (b, fb)) = decoders(alibi, rows)
    g = torch.Generator().manual_seed(rows)
    none = torch.empty(0)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).half().to(gpu)
    pad = torch.randint(0, 4, (rows, 1), generator=g).to(gpu)
    wide = torch.stack([pad, pad], 1)[:, 0]                            # the same values, strided
    x = rnd(rows, 6, 256)
    mask = D.alibi_mask(2, 6).to(gpu) if alibi else none
    for op in (a, b):
        op.forward(x, pad, none, True, True, True, mask)
    for t in range(3):
        x = rnd(rows, 1, 512)[:, :, ::2]                               # strided rows: the general call
        bias = D.alibi_mask(2, 7 + t)[:, -1:].contiguous().to(gpu) if alibi else none
        ya = a.forward(x.contiguous(), pad, none, True, True, False, bias).clone()
        yb = b.forward(x, wide, none, True, True, False, bias.float()).clone()
        assert torch.equal(ya, yb) and ya.shape == (rows, 1, 256) and a.step == b.step == 7 + t
        za = fa.forward(ya, True, True).clone()
        assert torch.equal(za, fb.forward(torch.stack([yb, yb], 2)[:, :, 0], True, True))
        assert torch.equal(fa.forward(ya, False, False), fb.forward(yb, True, False))
    x = x.contiguous()
    for bad in (dict(input=x.float()), dict(input=x[:, :, :128]), dict(input=x.expand(rows, 2, 256)), dict(input=x.cpu()),
                dict(pre_padding_len=pad.int()), dict(relative_attention_bias=rnd(2, 1, 3))):
        call = dict(dict(input=x, pre_padding_len=pad, reorder_state=none, pre_layernorm=True, add_residual=True,
                         first_pass=False, relative_attention_bias=bias), **bad)
        step = a.step
        with pytest.raises(RuntimeError, match="EET"):
            a.forward(**call)
        a.step = step
    a.step = cfg.max_full_seq
    with pytest.raises(RuntimeError, match="max_full_seq_len"):
        a.forward(x, pad, none, True, True, False, none)


@pytest.mark.parametrize("rows", [1, 32, 33])
@pytest.mark.parametrize("pre_layernorm", [True, False])
def test_feed_forward_refuses_a_host_input(monkeypatch, rows, pre_layernorm):
    """Before any buffer is asked for and any kernel sees the host pointer, at the sizes of both paths."""
    monkeypatch.setattr(ops, "_current_stream", lambda: 0)
    monkeypatch.setattr(ops, "check", lambda status, what: pytest.fail(f"{what} was called"))
    op = object.__new__(ops.GatedFeedForwardNetworkInt8)       # the constructor wants weights on a GPU
    op.desc = ops.MetaDesc(torch.float16, rows, 2, 64, 1, 1, activation_fn="silu", d_ff=64, is_int8=True)
    op.d_ff, op.beta, op.o_bias, op.cache_name = 64, None, None, "test_feed_forward_host_input"
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        op.forward(torch.zeros(rows, 1, 64, dtype=torch.float16), pre_layernorm, True)
    assert not any(key[1].type == "cpu" for key in ops.workspaces._bufs)


@pytest.mark.gpu
@pytest.mark.parametrize("alibi", [False, True])
@pytest.mark.parametrize("rows", [1, 5, 32, 33])
def test_all_layers_in_one_call(gpu, monkeypatch, alibi, rows):
    """Int8Decoder's steps through one library call for all layers and op by op: the same bits, caches and steps; op by
    op where a layer is not like the others, and from there on again in one call."""
    cfg = D.DecoderConfig(num_layers=3, hidden=256, heads=2, d_ff=704, vocab=64, alibi=alibi, max_batch=rows, max_prompt=8,
                          max_full_seq=16)
    sd, _ = D.random_state_dict(cfg, seed=6)
    one, each = (D.Int8Decoder(cfg, sd, device="cuda:0") for _ in range(2))
    whole, taken = ops.decode_layers, []

    def watched(*args):
        y = whole(*args)
        taken.append(y is not None)
        return y
    g = torch.Generator().manual_seed(rows)
    prompt, mask = torch.randint(0, 64, (rows, 6), generator=g).to(gpu), torch.ones(rows, 6, dtype=torch.long, device=gpu)
    mask[0, :2] = 0

    def step(i, ids, mask, reorder=None):
        out = []
        for model, form in ((one, watched), (each, lambda *a: None)):
            monkeypatch.setattr(ops, "decode_layers", form)
            model.reorder_state = torch.empty(0, dtype=torch.long) if reorder is None else reorder
            out.append(model.logits(ids, i < 0, mask).clone())
        assert torch.equal(*out)
        assert {a.step for m in (one, each) for a, _ in m.layers} == {6 + 1 + i if i >= 0 else 6}
        for (a, _), (b, _) in zip(one.layers, each.layers):
            if reorder is None:
                assert torch.equal(a._k, b._k) and torch.equal(a._v, b._v)
    step(-1, prompt, mask)
    for i in range(3):
        step(i, torch.randint(0, 64, (rows, 1), generator=g).to(gpu), mask if i < 2 else None)
    assert taken == [rows <= 32] * 3
    del taken[:]
    calls, first = [], one.layers[1][0]
    first.forward = lambda *a: calls.append(1) or type(first).forward(first, *a)       # a program's own
    step(3, prompt[:, :1], None)
    del first.forward
    assert taken == [False] and calls == [1]
    step(4, prompt[:, :1], None, torch.arange(rows, device=gpu).flip(0))               # a beam search's step
    assert taken[1:] == [False]
    first.step -= 1
    assert whole(one.layers, one.embed[prompt[:, :1]], None, None, None) is None       # the layers disagree


def two_decoders(alibi, rows):
    cfg = D.DecoderConfig(num_layers=3, hidden=256, heads=2, d_ff=704, vocab=64, alibi=alibi, max_batch=rows, max_prompt=8,
                          max_full_seq=16)
    sd, _ = D.random_state_dict(cfg, seed=7)
    return [D.Int8Decoder(cfg, sd, device="cuda:0") for _ in range(2)]


@pytest.mark.gpu
def test_a_failed_call_leaves_every_layer_where_it_was(gpu, monkeypatch):
    """No layer counts a token whose key and value it may not have; the call can be made again."""
    model, other = two_decoders(False, 3)
    g = torch.Generator().manual_seed(1)
    prompt, token = (torch.randint(0, 64, (3, n), generator=g).to(gpu) for n in (6, 1))
    for m in (model, other):
        m.logits(prompt, True)
    real = ops.check

    def failing(status, what=""):
        if what == "eet_decoder_int8_decode":
            raise RuntimeError("launch failed")
        real(status, what)
    monkeypatch.setattr(ops, "check", failing)
    with pytest.raises(RuntimeError, match="launch failed"):
        model.logits(token, False)
    assert [a.step for a, _ in model.layers] == [6, 6, 6]
    monkeypatch.setattr(ops, "check", real)
    got = model.logits(token, False).clone()
    assert torch.equal(got, other.logits(token, False)) and [a.step for a, _ in model.layers] == [7, 7, 7]


@pytest.mark.gpu
def test_layers_with_rotary_tables_of_their_own(gpu, monkeypatch):
    """A program may give an op another table (another base or scaling): each layer turns by its own."""
    one, each = two_decoders(False, 3)
    g = torch.Generator().manual_seed(2)
    prompt, token = (torch.randint(0, 64, (3, n), generator=g).to(gpu) for n in (6, 1))
    whole = ops.decode_layers
    for m in (one, each):
        m.logits(prompt, True)
        table = m.layers[1][0].rope_table
        m.layers[1][0].rope_table = table.flip(0).contiguous()
    a = one.logits(token, False).clone()
    monkeypatch.setattr(ops, "decode_layers", lambda *a: None)
    assert torch.equal(a, each.logits(token, False))
    each.layers[1][0].rope_table = table
    each.layers[0][0].step, each.layers[1][0].step, each.layers[2][0].step = 6, 6, 6
    assert not torch.equal(a, each.logits(token, False)) and whole is not ops.decode_layers
