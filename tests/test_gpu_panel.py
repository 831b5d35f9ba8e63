"""A prompt in panels (chpe_forward_tokens, and chpe_prefill past one block step) against the decode
steps of an engine that has neither (CHPE_BLOCK=0): the last position's logits and hidden state, and
the next decode step's logits, which read every cache row and recurrent state the panels left.

Prompt lengths at the edges of the block step (4, 8, 16), of the token tiles (32, 64, and 90 and 200 for those of
96 and 112), of the DeltaNet chunk (32) and of the panel (512), and odd ones.  The 2-norm bars: with the f32 cache each path is within 1e-5 of the 64-bit
result (f32 sums over 36 layers; measured 1e-6 to 8e-6), so they differ by less than 2e-5, with as
much again for the prompt; with the fp16 cache, rows whose f32 value lies within that distance of a
rounding boundary are stored one fp16 step apart (2^-11 of the value): measured 1e-5 to 2e-4, the
bars four times that.  An argmax may differ only where the two best logits are closer
than the bar.  (The 72B archives' panels: test_gpu_models.py, every tile against decode steps.)"""
import ctypes
import os
import shutil
import tempfile
import time

import numpy as np
import pytest

import chpe_amd as ca
import oracle as orc
from conftest import archive_path

pytestmark = pytest.mark.gpu

CASES = [  # archive kind, arch, vocabulary, fp16 cache, prompt lengths, bar
    (ca.PACK_3B_W4, 0, 151936, False, (4, 8, 9, 16, 17, 32, 33, 64, 65, 90, 129, 200, 512, 513, 577), 4e-5),
    (ca.PACK_3B_W4, 0, 151936, True, (5, 97, 600), 8e-4),
    (ca.PACK_3B_FP16_RAW, 0, 151936, False, (3, 31, 33, 64, 100, 515), 4e-5),
    (ca.PACK_3B_FP16_RAW, 0, 151936, True, (7, 130), 8e-4),
    (ca.PACK_9B_W4, 3, 248320, True, (4, 9, 16, 17, 32, 33, 65, 90, 100, 200, 513), 8e-4),
    (ca.PACK_9B_W4, 3, 248320, False, (5, 70), 8e-5),
    (ca.PACK_9B_W4, 1, 248320, False, (34, 70), 8e-5),
]


def rel(a, b):
    b = b.astype(np.float64)
    return float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b))


def engines(path, arch, rows, kv16, monkeypatch):
    monkeypatch.setenv("CHPE_BLOCK", "0")
    steps = ca.Engine(path, arch=arch, max_seq_len=rows, kv_f16=kv16)
    monkeypatch.delenv("CHPE_BLOCK")
    return ca.Engine(path, arch=arch, max_seq_len=rows, kv_f16=kv16), steps


@pytest.mark.timeout(600)
@pytest.mark.parametrize("kind,arch,vocab,kv16,lengths,bar", CASES)
def test_panels_match_decode_steps(kind, arch, vocab, kv16, lengths, bar, monkeypatch):
    e, steps = engines(archive_path(kind), arch, max(lengths) + 8, kv16, monkeypatch)
    try:
        for n in lengths:
            toks = np.random.default_rng(1000 * kind + n).integers(0, vocab, n).astype(np.uint32)
            am0, want = steps.forward_tokens(toks, want_logits=True)
            hid0 = steps.hidden()
            nxt0 = steps.decode_step(int(toks[0]), n)[1]
            steps.forward_tokens(toks)
            steps.time_steps(1)  # (the greedy loop's next step, from the device state the prompt left)
            gen0 = steps.logits()
            calls = [e.forward_tokens] + ([e.prefill] if n > 16 else [])
            for call in calls:
                am, got = call(toks, want_logits=True)
                hid = e.hidden()
                nxt = e.decode_step(int(toks[0]), n)[1]
                d = (rel(got, want), rel(hid, hid0), rel(nxt, nxt0))
                print(f"kind {kind} arch {arch} kv16 {kv16} n {n} {call.__name__}: logits {d[0]:.2e} hidden {d[1]:.2e} next {d[2]:.2e}",
                      flush=True)
                assert max(d) <= bar
                if am != am0:
                    assert want[am0] - want[am] <= bar * np.linalg.norm(want)
                    continue
                assert np.array_equal(call(toks, want_logits=True)[1].view(np.uint32), got.view(np.uint32))
                e.time_steps(1)
                assert rel(e.logits(), gen0) <= bar
    finally:
        e.close()
        steps.close()


def test_panel_break(w4_archive, monkeypatch):
    """forwardDecode's non-finite break (StepState::broken) in a panel: an infinite outlier weight
    in layer 1's down projection stops every token after that layer; the final norm and the LM head
    see that hidden state, as in the decode steps."""
    from test_gpu_nonfinite import inf_outlier_edit
    li = orc.layer_info(1, 1)
    off, b = inf_outlier_edit(w4_archive, li["down_proj"], li["down_tiles"])
    data = np.fromfile(w4_archive, dtype=np.uint8)
    data[off:off + 2] = np.frombuffer(b, np.uint8)
    fd, path = tempfile.mkstemp(suffix=".chpe", prefix="qwen2.5-3b-mod-", dir=os.path.dirname(str(w4_archive)))
    os.close(fd)
    data.tofile(path)
    try:
        e, steps = engines(path, 0, 64, False, monkeypatch)
        try:
            toks = np.random.default_rng(3).integers(0, 151936, 40).astype(np.uint32)
            am0, want = steps.forward_tokens(toks, want_logits=True)
            hid0, last0 = steps.hidden(), steps.last()
            am, got = e.forward_tokens(toks, want_logits=True)
            hid, last = e.hidden(), e.last()
            assert not np.isfinite(hid0).all()
            fin = np.isfinite(hid0)
            assert np.array_equal(np.isfinite(hid), fin) and rel(hid[fin], hid0[fin]) <= 4e-5
            assert np.array_equal(np.isnan(got), np.isnan(want)) and am == am0
            assert last["hidden_norm"] == last0["hidden_norm"] == np.inf
        finally:
            e.close()
            steps.close()
    finally:
        os.unlink(path)


@pytest.mark.timeout(300)
@pytest.mark.parametrize("kind,arch,vocab,kv16,at,bar", [
    (ca.PACK_3B_W4, 0, 151936, False, 21, 4e-5), (ca.PACK_3B_W4, 0, 151936, True, 21, 8e-4),
    (ca.PACK_9B_W4, 1, 248320, False, 23, 8e-5), (ca.PACK_9B_W4, 1, 248320, True, 23, 8e-4)])
def test_panel_nonfinite_row(kind, arch, vocab, kv16, at, bar, monkeypatch):
    """A token whose embedding row is not finite writes NaN keys and values into layer 0's cache; the
    attention of the tokens before it in the same tile of 16 rows (2 tokens of 8 heads, 4 of 4) must not
    meet them: a decode step that goes back to its position reads the rows before it, finite and as the
    decode steps left them.  (`at`: the last token of a tile.)"""
    bad, src = 1234, archive_path(kind)
    fd, path = tempfile.mkstemp(suffix=".chpe", prefix="qwen2.5-3b-mod-" if arch == 0 else "qwen3.5-9b-mod-",
                                dir=os.path.dirname(str(src)))
    os.close(fd)
    shutil.copyfile(src, path)
    cell = 4096 + bad // 16 * 17408 + 64 + 16384
    with open(path, "r+b") as f:  # 3B: the row's last outlier value; 9B: the tile's offset (16 tokens' rows)
        f.seek(cell + 560 + 16 * (bad % 16) + 14 if arch == 0 else cell + 36)
        f.write(np.float16(np.inf).tobytes() if arch == 0 else np.float32(np.inf).tobytes())
    try:
        e, steps = engines(path, arch, 64, kv16, monkeypatch)
        try:
            toks = np.random.default_rng(11).integers(2000, vocab, 40).astype(np.uint32)
            toks[at] = bad
            hid, nxt = [], []
            for x in (steps, e):
                x.forward_tokens(toks)
                hid.append(x.hidden())
                nxt.append(x.decode_step(2001, at)[1])
            fin = np.isfinite(nxt[0])
            assert not np.isfinite(hid[0]).any() and not np.isfinite(hid[1]).any()
            assert fin.sum() >= vocab - 16 and np.array_equal(np.isfinite(nxt[1]), fin)
            d = rel(nxt[1][fin], nxt[0][fin])
            print(f"arch {arch} kv16 {kv16}: the step at {at}: {d:.2e}", flush=True)
            assert d <= bar
        finally:
            e.close()
            steps.close()
    finally:
        os.unlink(path)


@pytest.mark.timeout(300)
@pytest.mark.parametrize("kind,gain", [(ca.PACK_3B_W4, 2.0 ** 16), (ca.PACK_3B_FP16_RAW, 2.0 ** 24)])
def test_panel_outlier_channel(kind, gain, monkeypatch):
    """One channel of every normalised input `gain` times the others, as the massive activations of real
    models: the other channels keep their bits, since every 128-column group has a scale of its own
    in the panels as in the decode steps.  (The weights of the channel's own group are zero in every
    projection that reads a normalised input, so the results depend on the other groups alone; with a
    scale per token the logits are 1e-3 apart.)"""
    src, raw, c0 = archive_path(kind), kind == ca.PACK_3B_FP16_RAW, 640
    fd, path = tempfile.mkstemp(suffix=".chpe", prefix="qwen2.5-3b-mod-", dir=os.path.dirname(str(src)))
    os.close(fd)
    shutil.copyfile(src, path)
    try:
        b = np.memmap(path, dtype=np.uint8, mode="r+")
        stride = 16384 if raw else 17408
        for l in range(36):
            li = orc.layer_info(0 if raw else 1, l)
            for name in ("q", "k", "v", "gate", "up"):
                rec, n = li[name + "_proj"], li[name + "_tiles"]
                t = b[4096 + rec * stride:4096 + (rec + n) * stride].reshape(n, stride)
                if raw:
                    t.view(np.float16).reshape(-1, 2048)[:, c0:c0 + 128] = 0
                    continue
                t[:, 64:16448].reshape(n, 16, 1024)[:, :, c0 // 2:c0 // 2 + 64] = 0x88
                cols = t[:, 16448 + 816:16448 + 832].copy().view(np.uint16)
                vals = t[:, 16448 + 560:16448 + 816].copy().view(np.float16).reshape(n, 16, 8)
                vals[np.broadcast_to((cols // 128 == c0 // 128)[:, None], vals.shape)] = 0
                t[:, 16448 + 560:16448 + 816] = vals.reshape(n, 128).view(np.uint8)
            for rec in (li["input_norm"], li["post_norm"]):
                at = 4096 + rec * stride + (0 if raw else 64) + 4 * (c0 + 77)
                b[at:at + 4] = (b[at:at + 4].copy().view(np.float32) * np.float32(gain)).view(np.uint8)
        b.flush()
        del b
        e, steps = engines(path, 0, 80, False, monkeypatch)
        try:
            toks = np.random.default_rng(5).integers(0, 151936, 70).astype(np.uint32)
            want, got = (x.forward_tokens(toks, want_logits=True)[1] for x in (steps, e))
            print(f"kind {kind} outlier channel: logits {rel(got, want):.2e}", flush=True)
            assert np.isfinite(want).all() and rel(got, want) <= 4e-5
        finally:
            e.close()
            steps.close()
    finally:
        os.unlink(path)


@pytest.mark.parametrize("call,n", [("forward_tokens", 3), ("forward_tokens", 20), ("prefill", 40)])
def test_refused_launch_is_an_error(w4_archive, call, n):
    """An error on the calling thread when the launches are done, as a refused launch leaves one (here: a device
    that does not exist), fails the call that it belongs to, in panels as in decode steps (n = 3); the call after it
    is right again."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    toks = np.random.default_rng(n).integers(0, 151936, n).astype(np.uint32)
    e = ca.Engine(w4_archive, arch=0, max_seq_len=64, kv_f16=False)
    try:
        want = getattr(e, call)(toks, want_logits=True)[1]
        assert hip.hipSetDevice(9999) != 0
        with pytest.raises(ca.EngineError):
            getattr(e, call)(toks)
        got = getattr(e, call)(toks, want_logits=True)[1]
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        e.close()


@pytest.mark.parametrize("mib", ["0", "40"])
def test_no_memory_for_panels(w4_archive, mib, monkeypatch):
    """Where the panels' buffers find no memory (a bound stands for it: none of them, the first few of them) the context
    still opens, holds none of them, and prompts run as before the panels: chpe_prefill in block steps of up to
    32 tokens, chpe_forward_tokens past 8 in decode steps, both bit for bit."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    toks = np.random.default_rng(9).integers(0, 151936, 75).astype(np.uint32)

    def mem_free():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    def run(fn):
        free = mem_free()
        e = ca.Engine(w4_archive, arch=0, max_seq_len=96, kv_f16=False)
        try:
            return free - mem_free(), fn(e)
        finally:
            e.close()

    def steps(e):
        return [e.decode_step(int(t), p)[1] for p, t in enumerate(toks[:20])][-1]

    def blocks(e):
        for i in (0, 32, 64):
            e.verify(toks[i:i + 32], i)
        return e.logits()

    run(steps)
    full, want = run(lambda e: (steps(e), blocks(e)))
    monkeypatch.setenv("CHPE_PANEL_MIB", mib)
    small, got = run(lambda e: (e.forward_tokens(toks[:20], want_logits=True)[1], e.prefill(toks, want_logits=True)[1]))
    for a, b in zip(got, want):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    print(f"context: {full >> 20} MiB, without panels {small >> 20}", flush=True)
    assert small < full - (64 << 20)


@pytest.mark.parametrize("n", [3, 6, 40])
def test_last_elapsed_is_a_tokens(w4_archive, n):
    """chpe_get_last_elapsed_ns after chpe_forward_tokens is one token's time (chpe_c_api.zig:107-111 after :61-63),
    whether the positions ran as decode steps, a block step or in panels: n times it is no more than the call,
    and no less than half of it."""
    e = ca.Engine(w4_archive, arch=0, max_seq_len=64, kv_f16=False)
    try:
        toks = np.random.default_rng(n).integers(0, 151936, n).astype(np.uint32)
        e.forward_tokens(toks)
        ratios = []
        for _ in range(9):
            t0 = time.perf_counter_ns()
            e.forward_tokens(toks)
            ratios.append(n * e.last()["elapsed_ns"] / (time.perf_counter_ns() - t0))
        assert 0.5 <= sorted(ratios)[4] <= 1.2, ratios
    finally:
        e.close()


@pytest.mark.parametrize("kind,arch,vocab", [(ca.PACK_3B_W4, 0, 151936), (ca.PACK_3B_FP16_RAW, 0, 151936), (ca.PACK_9B_W4, 3, 248320)])
def test_both_calls_take_the_same_route(kind, arch, vocab):
    """chpe_forward_tokens and chpe_prefill of the same tokens give the same bits from four positions on: logits, hidden
    state and the rows that the next step reads, around each of the rule's edges."""
    e = ca.Engine(archive_path(kind), arch=arch, max_seq_len=64, kv_f16=True)
    try:
        for n in (4, 8, 9, 12, 16, 17, 24, 32, 33):
            toks = np.random.default_rng(n).integers(0, vocab, n).astype(np.uint32)
            out = []
            for call in (e.forward_tokens, e.prefill):
                am, lg = call(toks, want_logits=True)
                out.append((am, lg, e.hidden(), e.decode_step(int(toks[0]), n)[1]))
            assert out[0][0] == out[1][0], n
            for a, b in zip(out[0][1:], out[1][1:]):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), n
    finally:
        e.close()
