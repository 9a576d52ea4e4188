"""The matrix recurrences at the sizes of real heads, against the plain torch functions (tests/emulated_ops.py)."""
import types

import pytest
import torch

from emulated_ops import EmulatedOps
from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def sequences(q_lens, starts, slots, device):
    cu, pos, seq = [0], [], []
    for i, (n, s) in enumerate(zip(q_lens, starts)):
        cu.append(cu[-1] + n)
        pos += list(range(s, s + n))
        seq += [i] * n
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=device)
    return types.SimpleNamespace(cu_q=i32(cu), positions=i32(pos), tok_seq=i32(seq), state_slots=i32(slots),
                                 num_seqs=len(q_lens), num_tokens=cu[-1], max_q_len=max(q_lens))


def close(a, b, tol):
    a, b = a.float().cpu(), b.float().cpu()
    assert torch.isfinite(a).all()
    assert (a - b).abs().max() <= tol * max(1.0, float(b.abs().max())), float((a - b).abs().max())


def test_normalisers_of_a_full_decode_batch():
    """A launch of many more blocks than the chip holds at once: every block needs the normaliser and the running maximum as
    they were before the step, also those that start when others have ended."""
    S, H, D, Dv = 64, 8, 128, 256
    hip, emu = HipOps(torch.float32, DEV), EmulatedOps(torch.float32)
    g = torch.Generator().manual_seed(3)
    buf = torch.randn(S, 2 * H * D + H * Dv + 2 * H, generator=g)
    state = torch.randn(S, H * D * Dv + H * D + H, generator=g) * 0.3
    args = ([1] * S, [5] * S, list(range(S)))
    cols = (0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * D + H * Dv + H)
    s1, s2 = state.clone().to(DEV), state.clone()
    o1 = hip.mlstm_scan(buf.to(DEV), *cols, H, D, Dv, 4.0, D ** -0.5, s1, sequences(*args, DEV), True)
    batch = sequences(*args, "cpu")
    batch.q_lens, batch.starts = args[0], args[1]
    o2 = emu.mlstm_scan(buf, *cols, H, D, Dv, 4.0, D ** -0.5, s2, batch, True)
    # 128 products of a head's read-out, over a divisor that is at least 1e-6 and mostly near one
    close(o1, o2, 2e-5)
    close(s1, s2, 2e-5)


Q_LENS, STARTS, SLOTS = [1, 31, 32, 33, 7, 100, 64], [0, 5, 0, 7, 300, 0, 9], [4, 0, 5, 2, 1, 6, 3]


def scan_case(mode, H, G, D, Dv, strong):
    """The call of ``mode`` on seeded inputs: (function of a kernel table, a state and a batch on a device) and the slot size."""
    g = torch.Generator().manual_seed(H * D + Dv)
    T = sum(Q_LENS)
    width = 2 * G * D + H * Dv
    src = torch.randn(T, width, generator=g)
    if "delta" in mode:                                    # (unit vectors, as the convolution in front of it makes them)
        heads = src[:, :2 * G * D].view(T, 2 * G, D)
        src[:, :2 * G * D] = (heads / heads.norm(dim=-1, keepdim=True)).flatten(1)
    gates = torch.randn(T, 2 * H, generator=g) * (4.0 if strong else 1.0)
    rates = torch.log(1.0 + 15.0 * torch.rand(H, generator=g))
    bias = torch.full((H,), 2.0 if strong else -3.0)
    log_decay = -torch.rand(T, H * D, generator=g) * (12.0 if strong else 0.1)
    if strong:
        log_decay[torch.rand(T, H * D, generator=g) < 0.05] = -1e4
    lower = torch.zeros(H * D) if strong else torch.rand(H * D, generator=g) * 0.9
    cols = (0, G * D, 2 * G * D)

    def call(ops, state, batch, device):
        d = lambda t: t.to(device)
        if mode == "decay":
            return ops.decay_scan(d(src), *cols, H, G, D, Dv, d(log_decay), 0.7, None, 0, state, batch, True)
        if mode == "delta":
            return ops.decay_scan(d(src), *cols, H, G, D, Dv, d(log_decay), 0.7, d(gates), H, state, batch, True)
        if mode == "delta, decay a head":
            return ops.head_delta_scan(d(src), *cols, H, G, D, Dv, d(gates), 0, H, d(rates), d(bias), state, batch, True)
        if mode == "state space":
            return ops.ssd_scan(d(src), 2 * G * D, G * D, 0, H, G, D, Dv, d(gates), H, d(rates), d(bias), d(rates), state,
                                batch, True)
        if mode == "forget":
            z = src.clone()
            z[:, G * D:2 * G * D] *= 30.0 if strong else 1.0
            return ops.forget_scan(d(z), 0, G * D, 2 * G * D, H, D, Dv, d(lower), state, batch, True, q_scale=0.5)
        buf = torch.cat([src, gates], 1)
        return ops.mlstm_scan(d(buf), *cols, width, width + H, H, D, Dv, 15.0, D ** -0.5, state, batch, True)
    return call, H * D * Dv + (H * D + H if mode == "lstm" else 0), torch.cat([src, gates], 1)


def lstm_read_outs(buf, state, H, D, Dv):
    """The matrix LSTM's read-outs in float64 and what their errors are measured by: with o = N / d, N = S^T q and d = |n q|
    or more, the terms that are added up for N over d, and o times those for n q over d (n q may cancel)."""
    buf, state = buf.double(), torch.nan_to_num(state.double())
    width, out, scale = 2 * H * D + H * Dv, [], []
    at = 0
    for n_tok, start, slot in zip(Q_LENS, STARTS, SLOTS):
        row = state[slot] * (start > 0)
        S, n, m = row[:H * D * Dv].view(H, Dv, D).transpose(1, 2), row[H * D * Dv:H * D * Dv + H * D].view(H, D), \
            row[H * D * Dv + H * D:H * D * Dv + H * D + H]
        for t in range(at, at + n_tok):
            q, k, v = buf[t, :H * D].view(H, D) * D ** -0.5, buf[t, H * D:2 * H * D].view(H, D), buf[t, 2 * H * D:width].view(H, Dv)
            i = 15 * torch.tanh(buf[t, width:width + H] / 15)
            f = torch.nn.functional.logsigmoid(15 * torch.tanh(buf[t, width + H:width + 2 * H] / 15))
            new = torch.maximum(f + m, i)
            keep, add, m = torch.exp(f + m - new), torch.exp(i - new), new
            S = keep[:, None, None] * S + add[:, None, None] * k[:, :, None] * v[:, None, :]
            n = keep[:, None] * n + add[:, None] * k
            d = torch.maximum((n * q).sum(-1).abs(), torch.exp(-m))[:, None] + 1e-6
            o = (S * q[:, :, None]).sum(1) / d
            out.append(o.flatten())
            scale.append(((S * q[:, :, None]).abs().sum(1) / d + o.abs() * (n * q).abs().sum(-1)[:, None] / d).flatten())
        at += n_tok
    return torch.stack(out), torch.stack(scale)


# heads of one, two, three and four blocks of 64 key channels, odd sizes, value channels that no slice divides
@pytest.mark.parametrize("H,G,D,Dv", [(2, 2, 128, 256), (3, 3, 20, 24), (2, 2, 72, 15), (1, 1, 200, 33), (2, 1, 256, 16), (4, 2, 64, 40)])
@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("mode", ["decay", "delta", "delta, decay a head", "state space", "forget", "lstm"])
def test_scan_in_chunks(mode, strong, H, G, D, Dv):
    """Sequences of one token up to several chunks, at their starts (their slots hold NaN) and going on, with weak decays and with
    ones that end a state at once."""
    if mode in ("forget", "lstm"):
        G = H
    hip, emu = HipOps(torch.float32, DEV), EmulatedOps(torch.float32)
    hip.SCAN_CHUNKS_FROM = hip.SCAN_CHUNKS_FROM_GROUPED = hip.SCAN_CHUNKS_FROM_MANY = 1
    call, size, buf = scan_case(mode, H, G, D, Dv, strong)
    g = torch.Generator().manual_seed(5)
    state = torch.randn(len(SLOTS), size + 3, generator=g) * 0.3
    for slot, start in zip(SLOTS, STARTS):
        if start == 0:
            state[slot] = float("nan")
    s1, s2 = state.clone().to(DEV), state.clone()
    o1 = call(hip, s1, sequences(Q_LENS, STARTS, SLOTS, DEV), DEV)
    host = sequences(Q_LENS, STARTS, SLOTS, "cpu")
    host.q_lens, host.starts = Q_LENS, STARTS
    o2 = call(emu, s2, host, "cpu")
    # both sides are float32: sums of up to 256 + 32 terms a chunk, as in the tests of the walk token by token
    if mode == "lstm":                                     # (2^-24 a rounding, chains of at most 64 of them on either side of the /)
        want, scale = lstm_read_outs(buf, state, H, D, Dv)
        assert ((o1.cpu().double() - want).abs() <= 1e-6 + 64 * 2.0 ** -24 * scale).all()
    else:
        close(o1, o2, 2e-5)
    close(s1[:, :size], s2[:, :size], 2e-5)
    assert torch.equal(torch.nan_to_num(s1.cpu()[:, size:], 9.0), torch.nan_to_num(state[:, size:], 9.0))


# a token in the middle of a block of 16, the last one of a chunk that is not full, the last one of a sequence
@pytest.mark.parametrize("H,G,D,Dv", [(2, 2, 72, 15), (4, 2, 64, 40)])
@pytest.mark.parametrize("what", ["value", "key", "decay"])
@pytest.mark.parametrize("mode", ["decay", "delta", "delta, decay a head", "state space", "forget", "lstm"])
def test_chunks_keep_infinities_and_nan_from_earlier_tokens(mode, what, H, G, D, Dv):
    """What is not finite in the walk token by token is not finite in chunks, and nothing else."""
    if mode in ("forget", "lstm"):
        G = H
    if mode == "forget" and what == "decay":
        what = "key"                                       # (its decays come from the keys)
    hip = HipOps(torch.float32, DEV)
    call, size, _ = scan_case(mode, H, G, D, Dv, False)
    inputs = dict(zip(call.__code__.co_freevars, (c.cell_contents for c in call.__closure__)))
    src, gates, log_decay = inputs["src"], inputs["gates"], inputs["log_decay"]
    first = [sum(Q_LENS[:i]) for i in range(len(Q_LENS))]
    for t in (first[5] + 40, first[5] + 75, first[3] + 32, first[4] + 6, first[6] + 18):
        if what == "value":
            src[t, 2 * G * D + 3] = float("inf")
        elif what == "key":
            src[t, G * D + 5] = float("nan")
        elif mode in ("decay", "delta"):
            log_decay[t, 7] = float("nan")
        else:
            gates[t, H if mode != "state space" else H] = float("nan")
    state = torch.randn(len(SLOTS), size, generator=torch.Generator().manual_seed(6)) * 0.3
    out, states = [], []
    for line in (1, 1 << 30):                              # in chunks, token by token
        hip.SCAN_CHUNKS_FROM = hip.SCAN_CHUNKS_FROM_GROUPED = hip.SCAN_CHUNKS_FROM_MANY = line
        states.append(state.clone().to(DEV))
        out.append(call(hip, states[-1], sequences(Q_LENS, STARTS, SLOTS, DEV), DEV))
    assert not torch.isfinite(out[1]).all()
    for a, b in (out, states):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
        if mode != "lstm" or a is not out[0]:              # (its read-outs are quotients: measured in test_scan_in_chunks)
            close(torch.nan_to_num(a, 0.0, 0.0, 0.0), torch.nan_to_num(b, 0.0, 0.0, 0.0), 2e-5)


def test_a_sequence_without_tokens_keeps_its_normaliser():
    """In chunks nothing is computed for it, so nothing may be copied to its slot either."""
    H, D, Dv, q_lens, starts = 2, 20, 24, [40, 0, 33], [0, 7, 3]
    hip = HipOps(torch.float32, DEV)
    hip.SCAN_CHUNKS_FROM = hip.SCAN_CHUNKS_FROM_MANY = 1
    g = torch.Generator().manual_seed(9)
    width = 2 * H * D + H * Dv
    buf = torch.randn(sum(q_lens), width + 2 * H, generator=g).to(DEV)
    state = torch.randn(3, H * D * Dv + H * D + H, generator=g).to(DEV)
    before = state.clone()
    hip.mlstm_scan(buf, 0, H * D, 2 * H * D, width, width + H, H, D, Dv, 15.0, D ** -0.5, state,
                   sequences(q_lens, starts, [2, 0, 1], DEV), True)
    assert torch.equal(state[0], before[0])
    assert (state[1:] != before[1:]).all(1).all()


@pytest.mark.parametrize("mode", ["decay", "delta", "delta, decay a head", "state space", "forget", "lstm"])
@pytest.mark.parametrize("order", [range(7), (5, 6, 3, 1, 2, 0, 4)])
def test_long_sequences_in_chunks_beside_short_ones(mode, order):
    """The two launches of such a step against all of it token by token; the long ones last and first."""
    H, G, D, Dv = (2, 2, 72, 33) if mode in ("forget", "lstm") else (4, 2, 64, 40)
    hip = HipOps(torch.float32, DEV)
    call, size, _ = scan_case(mode, H, G, D, Dv, False)
    lens, starts, slots = ([v[i] for i in order] for v in (Q_LENS, STARTS, SLOTS))
    batch = sequences(lens, starts, slots, DEV)
    state = torch.randn(len(slots), size, generator=torch.Generator().manual_seed(8)).to(DEV) * 0.3
    walked, both = state.clone(), state.clone()
    batch.q_lens = lens
    hip.SCAN_CHUNKS_FROM = hip.SCAN_CHUNKS_FROM_GROUPED = hip.SCAN_CHUNKS_FROM_MANY = 1 << 30
    want = call(hip, walked, batch, DEV)
    hip.SCAN_CHUNKS_FROM = hip.SCAN_CHUNKS_FROM_GROUPED = 40
    got = call(hip, both, batch, DEV)
    # (float32 in another order of sums, as against the plain functions above; the matrix LSTM's read-outs are quotients)
    close(got, want, 2e-5 if mode != "lstm" else 1e-3)
    close(both, walked, 2e-5)


def test_normalisers_of_a_long_portion():
    """More than 64 chunks, whose running maxima are put together 64 at a time, behind a context; against float64."""
    H, D, Dv, T = 2, 20, 24, 2100
    hip = HipOps(torch.float32, DEV)
    g = torch.Generator().manual_seed(11)
    width = 2 * H * D + H * Dv
    buf = torch.randn(T, width + 2 * H, generator=g) * 0.5
    buf[:, width + H:] += 4.0                              # (weak decays: a maximum is carried over many chunks)
    buf[3, width:width + H] = 14.0
    state = torch.randn(1, H * D * Dv + H * D + H, generator=g) * 0.3
    state[0, -H:] = 5.0
    s1 = state.clone().to(DEV)
    hip.mlstm_scan(buf.to(DEV), 0, H * D, 2 * H * D, width, width + H, H, D, Dv, 15.0, D ** -0.5, s1, sequences([T], [9], [0], DEV), True)
    row = state[0].double()
    S, n, m = row[:H * D * Dv].view(H, Dv, D), row[H * D * Dv:-H].view(H, D), row[-H:]
    for t in buf.double():
        k, v = t[H * D:2 * H * D].view(H, D), t[2 * H * D:width].view(H, Dv)
        i = 15 * torch.tanh(t[width:width + H] / 15)
        f = torch.nn.functional.logsigmoid(15 * torch.tanh(t[width + H:] / 15))
        new = torch.maximum(f + m, i)
        keep, add, m = torch.exp(f + m - new), torch.exp(i - new), new
        S, n = keep[:, None, None] * S + add[:, None, None] * v[:, :, None] * k[:, None], keep[:, None] * n + add[:, None] * k
    want = torch.cat([S.flatten(), n.flatten(), m])
    assert float((s1[0].double().cpu() - want).norm() / want.norm()) < 1e-5          # (chains of some hundred tokens)
