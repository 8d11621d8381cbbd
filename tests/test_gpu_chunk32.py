"""The fp32-input prefill's chunked form (what AUTO takes for fp32) against the
f64 oracle and against the token-sequential recurrence, at the sizes where
its tiles, its pipeline and its domain checks can go wrong.

The tolerance is the fp32 path's (rtol 1e-4, atol 1e-4 RMS).
"""
import numpy as np
import pytest
import torch

from gdr_cases import F32_TOL, Prefill, check_close

pytestmark = pytest.mark.gpu


def _check(w, o, fin, tag):
    ref_o, ref_f = w.oracle()
    mo = check_close(o.cpu().numpy(), ref_o, F32_TOL, f"{tag} o")
    mf = check_close(fin.cpu().numpy(), ref_f, F32_TOL, f"{tag} final state")
    print(f"{tag}: o {mo['normwise']:.2e}  final {mf['normwise']:.2e}", flush=True)
    return mo, mf


# chunks of 16 tokens, superblocks of 4 chunks, tiles of 32 rows, key widths
# padded to 32, 64 and 128, value tiles that end inside a scan wave's 16 rows
SHAPES = [
    dict(batch=1, heads=1, seq_len=1, d_k=4, d_v=4),
    dict(batch=2, heads=3, seq_len=79, d_k=32, d_v=32),
    dict(batch=1, heads=2, seq_len=80, d_k=20, d_v=36),
    dict(batch=3, heads=1, seq_len=81, d_k=64, d_v=64),
    dict(batch=1, heads=5, seq_len=127, d_k=36, d_v=12),
    dict(batch=1, heads=5, seq_len=64, d_k=36, d_v=12),
    dict(batch=1, heads=2, seq_len=65, d_k=100, d_v=52),
    dict(batch=2, heads=2, seq_len=129, d_k=128, d_v=128),
    dict(batch=1, heads=9, seq_len=200, d_k=128, d_v=256),
    dict(lengths=[0, 1, 16, 0, 31, 64, 200, 5, 0], heads=2, d_k=128, d_v=96, state_std=0.5),
    dict(lengths=[33, 79, 128], heads=3, d_k=64, d_v=32, state_std=0.02),
    # mostly short sequences, in one launch
    dict(lengths=[64, 65, 0, 3, 100, 7, 1, 64, 130, 33], heads=2, d_k=128, d_v=40, state_std=0.3),
    dict(lengths=[5, 40], heads=2, d_k=32, d_v=64),
    # just above the lengths that the recurrence keeps (96 tokens, 64 with d_k <= 32)
    dict(batch=1, heads=2, seq_len=97, d_k=100, d_v=52),
    dict(batch=2, heads=2, seq_len=112, d_k=128, d_v=128),
    dict(batch=1, heads=2, seq_len=113, d_k=68, d_v=36),
    dict(batch=2, heads=3, seq_len=65, d_k=32, d_v=32),
    dict(batch=1, heads=3, seq_len=97, d_k=36, d_v=32),
    dict(batch=1, heads=2, seq_len=144, d_k=20, d_v=36),
    dict(batch=3, heads=1, seq_len=145, d_k=64, d_v=64),
    dict(batch=1, heads=5, seq_len=191, d_k=36, d_v=12),
    dict(lengths=[0, 1, 97, 96, 31, 128, 200, 129, 0], heads=2, d_k=128, d_v=96, state_std=0.5),
    dict(lengths=[128, 129, 0, 160, 100], heads=3, d_k=64, d_v=32, state_std=0.02),
    dict(batch=1, heads=1, seq_len=3000, d_k=128, d_v=32, g_mean=-2.0, state_std=0.02),
    dict(batch=1, heads=2, seq_len=500, d_k=32, d_v=64, g_mean=5.0),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: ",".join(f"{k}={v}" for k, v in s.items()).replace(" ", ""))
def test_shapes(device, shape):
    w = Prefill(dtype=torch.float32, device=device, **shape)
    o, fin = w.run()
    mo, mf = _check(w, o, fin, str(shape))
    if w.d_k >= 64 and w.n_tok >= 1000:
        # no less accurate than the recurrence
        ro, rf = w.run(algo="recurrent")
        ref_o, ref_f = w.oracle()
        for x, y, ref in ((o, ro, ref_o), (fin, rf, ref_f)):
            e, er = (np.linalg.norm(t.double().cpu().numpy() - ref) for t in (x, y))
            assert e <= 1.05 * er, (e, er)


def test_unaligned_and_odd_shapes_keep_the_recurrence(device):
    """Widths that are no multiple of 4, and tensors 4 bytes off 16-byte
    alignment, at a length that the chunked form would take: RECURRENT's bits."""

    def off(x):
        buf = torch.empty(x.numel() + 1, device=device)
        buf[1:] = x.flatten()
        return buf[1:].reshape(x.shape)

    def check(w, tag):
        o, f = w.run()
        _check(w, o, f, tag)
        ro, rf = w.run(algo="recurrent")
        assert torch.equal(o, ro) and torch.equal(f, rf), tag

    kw = dict(batch=1, heads=2, seq_len=150, dtype=torch.float32, device=device, state_std=0.3)
    check(Prefill(d_k=30, d_v=12, **kw), "d_k 30")
    check(Prefill(d_k=32, d_v=10, **kw), "d_v 10")
    for name in ("q", "k", "v", "init"):
        w = Prefill(d_k=32, d_v=32, **kw)
        setattr(w, name, off(getattr(w, name)))
        check(w, f"{name} off alignment")


@pytest.mark.parametrize("d_k", [20, 32, 64, 128])
@pytest.mark.parametrize("g_mean", [1.0, -1.0, -4.0])
def test_error_against_64_bits_is_the_recurrences(device, d_k, g_mean):
    """From fast to slow decay, over several lengths, the chunked form's error
    is the recurrence's: 0.70 to 1.08 of it as measured (outputs and final
    states); samples of a few thousand values move the ratio by a few percent."""
    sums = np.zeros(4)
    for T in (129, 134, 144):
        w = Prefill(batch=4, heads=8, seq_len=T, d_k=d_k, d_v=64, dtype=torch.float32, device=device, g_mean=g_mean,
                    state_std=0.5)
        (o, f), (ro, rf), (xo, xf) = w.run(), w.run(algo="recurrent"), w.oracle()
        assert not torch.equal(o, ro)
        sums += [np.sum((a.double().cpu().numpy() - x) ** 2) for a, x in ((o, xo), (ro, xo), (f, xf), (rf, xf))]
    eo, ef = np.sqrt(sums[0] / sums[1]), np.sqrt(sums[2] / sums[3])
    print(f"d_k={d_k} g_mean={g_mean}: error ratio o {eo:.3f} final {ef:.3f}", flush=True)
    assert eo <= 1.15 and ef <= 1.15


@pytest.mark.parametrize("d_k", [32, 128])
def test_batch_invariant(device, d_k):
    """A sequence gives the same bits alone, in a pack of long sequences and in
    a pack whose average is short (which is launched in two parts)."""
    import rhizome_amd

    w = Prefill(lengths=[64, 200, 65, 17], heads=2, d_k=d_k, d_v=64, dtype=torch.float32, device=device,
                state_std=0.3)
    o, f = w.run()
    at = [(int(a), int(b)) for a, b in zip(w.cu[:-1], w.cu[1:])]
    for i, (a, b) in enumerate(at):
        for tail in (0, 80):  # alone, and followed by 80 empty sequences
            cu = torch.tensor([0, b - a] + [b - a] * tail, dtype=torch.int32, device=device)
            init = torch.cat([w.init[i:i + 1]] + [w.init[:1]] * tail)
            o1, f1 = rhizome_amd.prefill(w.q[a:b], w.k[a:b], w.v[a:b], w.g[a:b], w.beta[a:b], cu_seqlens=cu,
                                         initial_state=init)
            assert torch.equal(o1, o[a:b]) and torch.equal(f1[0], f[i])
            assert tail == 0 or torch.equal(f1[1:], init[1:])


@pytest.mark.parametrize("d_k,d_v", [(20, 12), (32, 96), (64, 40), (100, 64), (128, 128)])
@pytest.mark.parametrize("tail", [0, 300])
def test_short_sequences_are_the_recurrence(device, d_k, d_v, tail):
    """Sequences of up to 96 tokens (64 with d_k <= 32): the same bits in a
    pack, in a pack large enough for the recurrence's own launch (300 sequences
    more), in a dense batch and under RECURRENT."""
    import rhizome_amd

    w = Prefill(lengths=[96 if d_k > 32 else 64, 17, 0, 1, 33, 64] + [1] * tail, heads=2, d_k=d_k, d_v=d_v, dtype=torch.float32,
                device=device, state_std=0.3)
    o, f = w.run()
    ro, rf = w.run(algo="recurrent")
    assert torch.equal(o, ro) and torch.equal(f, rf)
    for i in (0, 1, 4):
        a, b = int(w.cu[i]), int(w.cu[i + 1])
        do, df = rhizome_amd.prefill(*(x[None, a:b].contiguous() for x in (w.q, w.k, w.v, w.g, w.beta)),
                                     initial_state=w.init[i:i + 1].contiguous())
        assert torch.equal(do[0], o[a:b]) and torch.equal(df[0], f[i])


# short and long sequences in turn, more than 256 workgroups of 32 rows, and a
# mean length of at most 64: the short ones go out in the recurrence's launch,
# the others in the chunked one
@pytest.mark.parametrize("d_k,d_v", [(32, 128), (64, 64), (128, 96)])
def test_pack_in_two_launches(device, d_k, d_v):
    import rhizome_amd

    lengths = [0, 1, 63, 64, 65, 200, 5, 97, 0, 70, 16, 96, 40, 0, 2, 1] * 4
    w = Prefill(lengths=lengths, heads=4, d_k=d_k, d_v=d_v, dtype=torch.float32, device=device, state_std=0.3)
    assert len(lengths) * w.heads * ((d_v + 31) // 32) > 256 and w.n_tok // len(lengths) <= 64
    o, f = w.run()
    _check(w, o, f, f"two launches d_k={d_k}")
    for i in range(len(lengths) - 16, len(lengths)):
        a, b = int(w.cu[i]), int(w.cu[i + 1])
        cu = torch.tensor([0, b - a], dtype=torch.int32, device=device)
        if b > a:
            o1, f1 = rhizome_amd.prefill(*(x[a:b] for x in (w.q, w.k, w.v, w.g, w.beta)), cu_seqlens=cu,
                                         initial_state=w.init[i:i + 1].contiguous())
            assert torch.equal(o1, o[a:b]) and torch.equal(f1[0], f[i])
        else:
            assert torch.equal(f[i], w.init[i])


@pytest.mark.parametrize("m", [1, 16, 21, 64])
def test_reset_forgets_history(device, m):
    """alpha = 0 at position m: outputs from m on and final states are the same
    numbers whatever came before."""
    import rhizome_amd

    w = Prefill(batch=2, heads=2, seq_len=150, d_k=128, d_v=32, dtype=torch.float32, device=device, state_std=0.5)
    h = Prefill(batch=2, heads=2, seq_len=150, d_k=128, d_v=32, dtype=torch.float32, device=device, state_std=0.02,
                seed=1)

    def run(a, b):
        mix = [torch.cat([w.shaped(x)[:, :m], w.shaped(y)[:, m:]], 1).contiguous()
               for x, y in ((a.q, b.q), (a.k, b.k), (a.v, b.v), (torch.exp(a.g), torch.exp(b.g)), (a.beta, b.beta))]
        mix[3][:, m] = 0.0
        return rhizome_amd.prefill(mix[0], mix[1], mix[2], None, mix[4], alpha=mix[3], initial_state=a.init)

    (o1, f1), (o2, f2) = run(w, w), run(h, w)
    assert torch.equal(o1[:, m:], o2[:, m:]) and torch.equal(f1, f2)
    assert not torch.equal(o1[:, :m], o2[:, :m])


def _leave(w, case, t, h):
    if case == "beta |k|^2 above 2":
        w.k[t, h] *= 3.0
    elif case == "beta -0.5":
        w.beta[t, h] = -0.5
    elif case == "alpha 1.05":
        w.g[t, h] = float(np.log(1.05))
    elif case == "v inf":
        w.v[t, h, 3] = float("inf")
    elif case == "v nan in the second row half":
        w.v[t, h, 20] = float("nan")
    elif case == "q nan":
        w.q[t, h, 5] = float("nan")
    elif case == "k nan":
        w.k[t, h, 1] = float("nan")
    elif case == "beta nan":
        w.beta[t, h] = float("nan")
    elif case == "gate nan":
        w.g[t, h] = float("nan")
    elif case == "v 3e38":  # finite, but its sums overflow
        w.v[t - 8:t + 6, h, 40] = 3e38
    else:
        raise ValueError(case)


CASES = ["beta |k|^2 above 2", "beta -0.5", "alpha 1.05", "v inf", "v nan in the second row half", "q nan", "k nan",
         "beta nan", "gate nan", "v 3e38"]


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("d_k", [128, 64, 24])
def test_out_of_domain_is_the_recurrence(device, case, in_place, d_k):
    """Inputs outside the op's domain or not finite, at the last token of a
    16-token chunk or at the first of a partial one, in one head: every other
    (sequence, head) is unchanged, and the head's tiles equal the recurrence
    bit for bit or the chunked result where they hold no such value (a value
    row's tile), also when the state is updated in place."""
    kw = dict(heads=2, d_k=d_k, d_v=64, lengths=[47, 102], dtype=torch.float32, device=device, state_std=0.1)
    w, plain = Prefill(**kw), Prefill(**kw)
    if "3e38" in case:
        w.q *= 1e3
        plain.q *= 1e3
    _leave(w, case, 47 + 31 if "row" in case else 47 + 96, 1)
    want_o, want_f = plain.run()

    def run(**k):
        import rhizome_amd

        init = w.init.clone()
        fin = init if in_place else None
        return rhizome_amd.prefill(w.q, w.k, w.v, w.g, w.beta, cu_seqlens=w.cu_dev, initial_state=init,
                                   final_state=fin, **k)

    (o, f), (ro, rf) = run(), run(algo="recurrent")
    bits = lambda x: x.contiguous().view(torch.int32)  # noqa: E731  (NaN compares equal to itself)
    other = torch.ones(o.shape[:2], dtype=torch.bool, device=device)
    other[47:, 1] = False
    assert torch.equal(o[other], want_o[other]) and torch.equal(f[0], want_f[0]) and torch.equal(f[1, 0], want_f[1, 0])
    touched = 0
    for i0 in (0, 32):  # the head's two tiles
        a, r = o[47:, 1, i0:i0 + 32], ro[47:, 1, i0:i0 + 32]
        fa, fr = f[1, 1, i0:i0 + 32], rf[1, 1, i0:i0 + 32]
        same = torch.equal(torch.isnan(a), torch.isnan(r)) and torch.equal(bits(a.nan_to_num()), bits(r.nan_to_num())) \
            and torch.equal(bits(fa.nan_to_num()), bits(fr.nan_to_num()))
        touched += same
        if not same:  # a tile without the value: the chunked result
            assert torch.equal(a, want_o[47:, 1, i0:i0 + 32]) and torch.equal(fa, want_f[1, 1, i0:i0 + 32])
    assert touched >= 1


@pytest.mark.parametrize("t", [0, 15, 63, 64, 127, 128, 250, 255, 256, 278, 280])
@pytest.mark.parametrize("d_k", [128, 64, 32])
def test_leaves_the_domain_anywhere(device, t, d_k):
    """An input outside the domain in the first 64 tokens, where the pipeline
    ends at once, and in every later superblock of 64: the recurrence's results
    in its head, unchanged ones elsewhere, with the state updated in place too."""
    T = 250 if t == 0 else 281  # 4 superblocks or 5, and a last chunk that is not full
    kw = dict(heads=2, d_k=d_k, d_v=40, batch=1, seq_len=T, dtype=torch.float32, device=device, state_std=0.1)
    w, plain = Prefill(**kw), Prefill(**kw)
    t = min(t, T - 1)
    w.beta[t, 0] = -0.25
    want_o, want_f = plain.run()
    ro, rf = w.run(algo="recurrent")
    o, f = w.run()
    w.init = w.init.clone()
    oi, fi = w.run(final_state=w.init)
    assert torch.equal(o, oi) and torch.equal(f, fi)
    assert torch.equal(o[:, 0], ro[:, 0]) and torch.equal(f[:, 0], rf[:, 0])
    assert torch.equal(o[:, 1], want_o[:, 1]) and torch.equal(f[:, 1], want_f[:, 1])


def test_more_workgroups_than_a_grid_holds(device):
    """A pack of one-token sequences and a long one after them, in more
    workgroups than a grid of 512 threads each holds (2^32 / 512): one token's
    output and state in closed form, the long sequence as when run alone."""
    import rhizome_amd

    N, H, dk, dv, T = 1 << 18, 16, 4, 36, 81
    gen = torch.Generator(device=device).manual_seed(7)
    rand = lambda *s: torch.randn(*s, generator=gen, device=device)  # noqa: E731
    q, k, v = rand(N + T, H, dk), rand(N + T, H, dk), rand(N + T, H, dv)
    k /= k.norm(dim=-1, keepdim=True)
    g, beta = -torch.nn.functional.softplus(rand(N + T, H)), torch.sigmoid(rand(N + T, H))
    cu = torch.cat([torch.arange(N + 1), torch.tensor([N + T])]).int().to(device)
    o, fin = rhizome_amd.prefill(q, k, v, g, beta, cu_seqlens=cu)
    bv = beta[:N, :, None] * v[:N]
    # sums of four products of N(0, 1) values in fp32
    assert float((o[:N] - bv * (k[:N] * q[:N]).sum(-1, keepdim=True)).abs().max()) < 1e-4
    assert float((fin[:N] - bv[..., None] * k[:N, :, None]).abs().max()) < 1e-5
    alone = torch.tensor([0, T], dtype=torch.int32, device=device)
    o1, f1 = rhizome_amd.prefill(q[N:], k[N:], v[N:], g[N:], beta[N:], cu_seqlens=alone)
    assert torch.equal(o[N:], o1) and torch.equal(fin[N], f1[0])
