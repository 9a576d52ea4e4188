"""Kernels of a step of few tokens that ask for a whole row at once, at the edges of the rows they can hold, against the plain torch
functions; slots of sequences at their start hold NaN."""
import pytest
import torch

from servelab_amd.parts.base import RotaryTables
from test_vekanex_kernels_gpu import DEV, close, fake_batch, tables

pytestmark = pytest.mark.gpu
# a bfloat16 result differs by one rounding at most (2^-8 of it), a float32 one by the order of its sums
BAR = {torch.float32: 3e-6, torch.bfloat16: 8e-3}


# rows of up to 64 channels, of each number of them a lane, one more; slices and latent rows likewise
@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 256, 257, 512, 513])
@pytest.mark.parametrize("dtype", list(BAR))
def test_norms_of_heads_and_slices(n, dtype):
    hip, emu = tables(dtype)
    g = torch.Generator().manual_seed(n)
    T, H = 3, 2
    o, gate = torch.randn(T, H * n, generator=g), torch.randn(T, 5 + H * n, generator=g)
    for per_head in (True, False):
        w = 1 + 0.3 * torch.randn((H * n) if per_head else n, generator=g)
        for z, kw in ((None, {}), (gate, dict(activation="silu")), (gate, dict(activation="silu", gate_first=True)), (gate, {})):
            got = hip.head_norm_gate(o.to(DEV), H, n, w.to(DEV), per_head, 1e-5, None if z is None else z.to(DEV), 5, **kw)
            close(got, emu.head_norm_gate(o, H, n, w, per_head, 1e-5, z, 5, **kw), BAR[dtype])
    D, R, page = 8, 4, 16
    buf, gain = torch.randn(T, 3 + n + R, generator=g).to(dtype), 1 + 0.2 * torch.randn(n, generator=g)
    q_rows, slots = torch.randn(T, H * (D + R), generator=g).to(dtype), torch.tensor([5, 17, 0], dtype=torch.int32)
    k1, q1 = torch.zeros(2, 1, page, n + R).to(dtype), torch.zeros(T, H * (n + R)).to(dtype)
    k2, q2 = k1.to(DEV), q1.to(DEV)
    ang = torch.rand(T, R // 2, generator=g)
    tb = RotaryTables(torch.cos(ang), torch.sin(ang))
    emu.latent_store(buf, H, D, R, n, 3, R, gain, 1e-5, tb, slots, k1, page, q1, q_rows=q_rows)
    hip.latent_store(buf.to(DEV), H, D, R, n, 3, R, gain.to(DEV), 1e-5, RotaryTables(tb.cos.to(DEV), tb.sin.to(DEV)), slots.to(DEV), k2, page,
                     q2, q_rows=q_rows.to(DEV))
    close(k2, k1, BAR[dtype])
    close(q2, q1, BAR[dtype])
    close(hip.slice_rmsnorm(buf.to(DEV), 3, n, gain.to(DEV), 1e-5), emu.slice_rmsnorm(buf, 3, n, gain, 1e-5), BAR[dtype])


# steps of 64 tokens and 65; rows of 4,096 values of q and k and above, of 1,024 of v and above; sizes that are no powers of two; no keys of
# their own; alone, and behind a convolution of four taps (its row of up to 4,096 channels, and above), of three, of one; single tokens,
# whose slots move on in the launch, and longer ones.  (Without a norm: the kernel of a wavefront a head.)
@pytest.mark.parametrize("T,H,G,D,Dv", [(1, 16, 2, 128, 128), (64, 2, 1, 16, 8), (65, 2, 1, 16, 8), (3, 31, 1, 128, 24), (2, 30, 3, 128, 40),
                                        (5, 5, 3, 20, 341), (4, 5, 3, 20, 342), (3, 24, 8, 96, 128), (2, 3, 2, 9, 7)])
@pytest.mark.parametrize("taps", [0, 1, 3, 4])
def test_rows_of_a_step(T, H, G, D, Dv, taps):
    hip, emu = tables(torch.float32)
    g = torch.Generator().manual_seed(H + T)
    page, width = 16 if T % 2 else 24, (H + G) * D + G * Dv
    rot = D // 4 * 2
    buf = torch.randn(T, width + 3, generator=g)
    ang = torch.rand(T, rot // 2, generator=g) * 6
    tb = RotaryTables(torch.cos(ang), torch.sin(ang))
    tbd = RotaryTables(tb.cos.to(DEV), tb.sin.to(DEV))
    slots = torch.randperm(page * 5, generator=g)[:T].to(torch.int32)
    qg, kg = 1 + 0.2 * torch.randn(H * D, generator=g), 1 + 0.2 * torch.randn(G * D, generator=g)
    for lens in ([1] * T, [T]) if taps else ([1] * T,):
        for norm in (True, False):
            k1, v1 = torch.zeros(5, G, page, D), torch.zeros(5, G, Dv, page)
            k2, v2 = k1.to(DEV), v1.to(DEV)
            conv = conv_d = None
            if taps:
                starts, used = [3 * (i % 2) for i in range(len(lens))], torch.randperm(len(lens) + 1, generator=g)[:len(lens)].tolist()
                s1 = torch.randn(len(lens) + 1, 2 + (taps - 1) * width, generator=g)
                for s, at in zip(starts, used):
                    if s == 0:
                        s1[at] = float("nan")
                s2, w = s1.to(DEV), torch.randn(width, taps, generator=g)
                conv, conv_d = (w, s1, 1, fake_batch(lens, starts, used, "cpu"), True), (w.to(DEV), s2, 1, fake_batch(lens, starts, used, DEV), True)
            args = (1e-5, rot)
            want = emu.projnorm_rope_store(buf, H, G, D, Dv, qg if norm else None, kg if norm else None, *args, tb, slots, k1, v1, page, conv=conv)
            got = hip.projnorm_rope_store(buf.to(DEV), H, G, D, Dv, qg.to(DEV) if norm else None, kg.to(DEV) if norm else None, *args, tbd,
                                          slots.to(DEV), k2, v2, page, conv=conv_d)
            close(got, want, BAR[torch.float32])
            close(k2, k1, BAR[torch.float32])
            close(v2, v1, BAR[torch.float32])
            if taps:
                assert torch.equal(s2.cpu().nan_to_num(9.0), s1.nan_to_num(9.0))


# no trip of eight k-steps, one, one and a k-step, two
@pytest.mark.parametrize("K", [32, 224, 256, 288, 512])
@pytest.mark.parametrize("T", [1, 4])
def test_trips_of_head_products(K, T):
    hip, emu = tables(torch.bfloat16)
    g = torch.Generator().manual_seed(K)
    heads, N = 3, 48
    x, A = torch.randn(T, heads * K, generator=g).bfloat16(), (torch.randn(heads, N, K, generator=g) * K ** -0.5).bfloat16()
    close(hip.head_products(x.to(DEV), 0, heads, K, A.to(DEV)), emu.head_products(x, 0, heads, K, A), BAR[torch.bfloat16])
