"""Beam search over shared cache rows (eet_mmha_decode_beams): against the cache reorder followed by the ordinary
call, which moves the same rows -- the same sums in the same order, so the outputs are equal bit for bit."""
import copy
import threading

import numpy as np
import pytest
import torch

from eet_amd import decoder as D
from eet_amd._lib import check, lib
from gpu_util import mmha, stream


def test_argument_errors():
    L = lib()
    buf = np.zeros(4096, np.uint8)
    p, q = buf.ctypes.data, buf.ctypes.data + 1024

    def call(k=p, rows_in=p, rows_out=q, reorder=p, B=1, H=1, dh=64, step=4, cap=8):
        return L.eet_mmha_decode_beams(p, k, k, 0, p, p, p, None, None, B, H, dh, step, cap, None, rows_in, rows_out,
                                       reorder, None, 0, None)
    assert call(k=None) == -1
    assert call(rows_out=None) == -1
    assert call(rows_in=q) == -1                     # a reorder may not read the table it writes
    assert call(reorder=None) == -1                  # without one the table is updated in place
    assert call(reorder=None, rows_in=None) == -1
    assert call(B=65, H=32, dh=128, cap=4096) == -2  # 2 GiB of K cache is the largest
    assert call(step=9) == -1
    assert call(dh=40) == -2
    assert L.eet_kv_cache_gather_rows(p, p, p, p, p, 1, 1, 64, 4, 8, None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,dh,first,cap,padded,alibi", [
    (2, 1, 32, 1, 8, False, False),          # from a one-row prompt on
    (5, 3, 96, 30, 40, True, True),          # idle lanes, padding, bias
    (16, 8, 64, 255, 262, True, False),      # one workgroup per (sequence, head), whole turns of the ring and a row
    (3, 8, 128, 1021, 1030, False, True),    # several splits
    (260, 1, 32, 700, 704, False, False),    # more names per workgroup than lanes
    (8, 32, 128, 2058, 2064, True, False),   # 64 rows to a stream: the ring of four by the plan itself
])
def test_rows_by_name_equal_moved_rows(gpu, B, H, dh, first, cap, padded, alibi):
    g = torch.Generator().manual_seed(B * 1000 + dh)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).half().to(gpu)
    L = lib()
    kc, vc = rnd(B, H, cap, dh), rnd(B, H, cap, dh)              # rows by name: never moved
    km, vm = kc.clone(), vc.clone()                              # moved before every call
    tables = [torch.zeros(B, cap, dtype=torch.int32, device=gpu) for _ in range(2)]
    names = None
    pad = torch.tensor([(7 * b) % max(first, 1) for b in range(B)], device=gpu) if padded else None
    rope = torch.empty(cap, dh, device=gpu)
    check(L.eet_rope_table(rope.data_ptr(), cap, dh, stream()))
    for step, reordered in zip(range(first + 1, cap + 1), [True, True, False, True, True, False, True, True, True]):
        q, k, v = rnd(B, H * dh), rnd(B, H * dh), rnd(B, H * dh)
        bias = rnd(H, step) if alibi else None
        order = None
        if reordered:
            order = torch.randint(0, B, (B,), generator=g)
            order[B // 2] = B if step % 2 else -1                # out of range: the beam keeps its own rows
            order = order.to(gpu)
            k2, v2 = torch.zeros_like(km), torch.zeros_like(vm)
            check(L.eet_kv_cache_reorder(km.data_ptr(), vm.data_ptr(), k2.data_ptr(), v2.data_ptr(), order.data_ptr(),
                                         B, H, dh, step - 1, cap, stream()))
            km, vm = k2, v2
        row = rope[step - 1]
        want = mmha(q, k, v, km, vm, step, pad, bias, rope_row=row)
        if names is None and order is None:
            got = mmha(q, k, v, kc, vc, step, pad, bias, rope_row=row)
        else:
            out = names if order is None else tables[1 if names is tables[0] else 0]
            got = torch.empty_like(want)
            need = L.eet_mmha_decode_workspace(B, H, dh, step)
            ws = torch.empty(max(need // 4, 1), device=gpu)
            check(L.eet_mmha_decode_beams(
                q.data_ptr(), k.data_ptr(), v.data_ptr(), 0, kc.data_ptr(), vc.data_ptr(), got.data_ptr(),
                bias.data_ptr() if alibi else None, pad.data_ptr() if padded else None, B, H, dh, step, cap,
                row.data_ptr(), names.data_ptr() if names is not None else None, out.data_ptr(),
                order.data_ptr() if order is not None else None, ws.data_ptr(), ws.numel() * 4, stream()))
            names = out
        assert torch.equal(got, want), f"step {step}"
        if names is not None:
            ks, vs = torch.zeros_like(kc), torch.zeros_like(vc)
            check(L.eet_kv_cache_gather_rows(kc.data_ptr(), vc.data_ptr(), ks.data_ptr(), vs.data_ptr(),
                                             names.data_ptr(), B, H, dh, step, cap, stream()))
            assert torch.equal(ks[:, :, :step], km[:, :, :step]) and torch.equal(vs[:, :, :step], vm[:, :, :step])


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 40])          # one library call per op, separate launches
def test_op_settles_its_cache(gpu, rows):
    """A call that cannot name rows (fewer sequences than the prompt had) and a read of the cache in between give
    what rows that moved on every reorder give."""
    cfg = D.DecoderConfig(num_layers=1, hidden=256, heads=4, d_ff=704, vocab=64, max_batch=rows, max_prompt=8,
                          max_full_seq=32)
    sd, _ = D.random_state_dict(cfg, seed=3)
    a, b = (D.Int8Decoder(cfg, sd, device="cuda:0") for _ in range(2))
    g = torch.Generator().manual_seed(1)
    ids = torch.randint(0, 64, (rows, 6), generator=g).to(gpu)
    assert torch.equal(a.logits(ids, True), b.logits(ids, True))
    for t, n in enumerate([rows, rows, rows - 1, rows - 1, rows]):
        order = torch.randint(0, rows, (rows,), generator=g).to(gpu) if t != 3 else torch.empty(0, dtype=torch.long)
        ids = torch.randint(0, 64, (n, 1), generator=g).to(gpu)
        a.reorder_state = b.reorder_state = order
        la, lb = a.logits(ids, False), b.logits(ids, False)
        assert torch.equal(la, lb)
        ka = b.layers[0][0].k_cache                # b settles after every step, a only when it must
        assert b.layers[0][0]._rows is None and ka.shape[0] == rows
    step = a.layers[0][0].step
    assert torch.equal(a.layers[0][0].k_cache[: rows - 1, :, :step], b.layers[0][0].k_cache[: rows - 1, :, :step])


@pytest.mark.gpu
@pytest.mark.parametrize("ring", [2, 4])
@pytest.mark.parametrize("threads,nsplit", [(256, 1), (512, 3), (1024, 2)])
@pytest.mark.parametrize("B,H,dh,first,cap,padded,alibi", [(4, 3, 128, 700, 706, True, True), (3, 2, 96, 411, 416, False, False),
                                                           (5, 2, 64, 1500, 1504, False, True), (2, 3, 32, 3001, 3005, True, False)])
def test_every_form_of_the_kernel(gpu, tuning, ring, threads, nsplit, B, H, dh, first, cap, padded, alibi):
    """Both depths of the ring, whose slots hold the names requested a turn ahead, at every width of a workgroup and
    with the time axis split: several turns and a ragged last one."""
    tuning("EET_MMHA_THREADS", threads)
    tuning("EET_MMHA_UNROLL", ring)
    tuning("EET_MMHA_NSPLIT", nsplit)
    test_rows_by_name_equal_moved_rows(gpu, B, H, dh, first, cap, padded, alibi)


def beam_decoders(rows, steps):
    cfg = D.DecoderConfig(num_layers=2, hidden=256, heads=4, d_ff=704, vocab=64, max_batch=rows, max_prompt=8,
                          max_full_seq=8 + steps)
    sd, _ = D.random_state_dict(cfg, seed=3)
    a, b = (D.Int8Decoder(cfg, sd, device="cuda:0") for _ in range(2))
    g = torch.Generator().manual_seed(rows)
    ids = torch.randint(0, 64, (rows, 8), generator=g).cuda()
    assert torch.equal(a.logits(ids, True), b.logits(ids, True))
    calls = [(torch.randint(0, 64, (rows, 1), generator=g).cuda(), torch.randint(0, rows, (rows,), generator=g).cuda())
             for _ in range(steps)]

    def step(model, t):
        ids, model.reorder_state = calls[t]
        return model.logits(ids, False)
    return a, b, step


@pytest.mark.gpu
def test_cache_read_on_another_stream(gpu):
    """While the ops' stream is far behind: the rows that the reader gets are those of the finished step, and the
    steps after it go on from them."""
    a, b, step = beam_decoders(5, 6)
    side = torch.cuda.Stream()
    for t in range(6):
        torch.cuda._sleep(20_000_000)
        la = step(a, t).clone()
        if t % 2 == 0:
            with torch.cuda.stream(side):
                k = a.layers[1][0].k_cache.clone()
                v = a.layers[0][0].v_cache.clone()
            side.synchronize()
        assert torch.equal(la, step(b, t))
        if t % 2 == 0:
            n = b.layers[0][0].step
            assert torch.equal(k[:, :, :n], b.layers[1][0].k_cache[:, :, :n])
            assert torch.equal(v[:, :, :n], b.layers[0][0].v_cache[:, :, :n])


@pytest.mark.gpu
def test_cache_read_from_another_thread(gpu):
    """A thread that looks at the caches all the time, on a stream of its own, changes no step."""
    steps = 60
    a, b, step = beam_decoders(4, steps)
    want = [step(b, t).clone() for t in range(steps)]
    done, seen = threading.Event(), []

    def watch():
        with torch.cuda.stream(torch.cuda.Stream()):
            while not done.is_set():
                seen.append(tuple(a.layers[len(seen) % 2][0].k_cache.shape))
    reader = threading.Thread(target=watch)
    reader.start()
    try:
        got = [step(a, t).clone() for t in range(steps)]
    finally:
        done.set()
        reader.join()
    assert seen and all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.gpu
def test_copied_op(gpu):
    """A deep copy taken in mid-search goes on by itself."""
    a, b, step = beam_decoders(3, 4)
    for t in range(2):
        step(a, t), step(b, t)
    c = copy.deepcopy(a)
    for t in (2, 3):
        want = step(b, t).clone()
        assert torch.equal(step(a, t), want) and torch.equal(step(c, t), want)


@pytest.mark.gpu
def test_cache_of_a_sequence_set_back(gpu):
    """Setting `step` back loses no row: what a reader finds behind it are the rows that moved on every reorder."""
    a, b, step = beam_decoders(4, 6)
    for t in range(5):
        step(a, t), step(b, t)
        b.layers[0][0].k_cache, b.layers[1][0].k_cache        # settles after every step
    for model in (a, b):
        for attn, _ in model.layers:
            attn.step = 9
    ids = torch.arange(4).view(4, 1).cuda()                   # a call over named rows, without a reorder, in between
    for model in (a, b):
        model.reorder_state = torch.empty(0, dtype=torch.long)
        model.logits(ids, False)
    for (x, _), (y, _) in zip(a.layers, b.layers):
        assert x.step == y.step == 10
        assert torch.equal(x.k_cache[:, :, :13], y.k_cache[:, :, :13])
        assert torch.equal(x.v_cache[:, :, :13], y.v_cache[:, :, :13])
