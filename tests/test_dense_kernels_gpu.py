"""The dense decoders' kernels at the edges of their tiles, splits and routes,
against float64."""

import math

import pytest
import torch

from llmapigateway_amd import ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
D = 128


def _pages(lens, Hkv, BS, fp8, seed, most=None):
    """Pages of random keys and values, shuffled tables wide enough for a
    context of ``most``, and the same as float64 values."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    B = len(lens)
    width = -(-max(lens + [most or 0]) // BS)
    NB = B * -(-max(lens) // BS) + 3
    tables = torch.zeros(B, width, dtype=torch.int32, device=DEV)
    used = -(-max(lens) // BS)
    tables[:, :used] = torch.randperm(NB, generator=g, device=DEV)[: B * used].view(B, used).int()
    kv, scales, wide = [], [], []
    for _ in range(2):
        x = torch.randn(NB, Hkv, BS, D, generator=g, device=DEV)
        if fp8:
            x = (x * 64).to(torch.float8_e4m3fn)
            s = torch.rand(NB, Hkv, BS, generator=g, device=DEV) * 0.02 + 0.001
            kv.append(x.view(torch.uint8))
            scales.append(s)
            wide.append(x.double() * s.double().unsqueeze(-1))
        else:
            kv.append(x.bfloat16())
            scales.append(None)
            wide.append(kv[-1].double())
    return kv, scales, wide, tables


def _softmax_rows(q, k, v):
    """q [G, D], k and v [L, D] of one kv head, float64."""
    return (q @ k.T / math.sqrt(D)).softmax(-1) @ v


# 16 (bf16) and 32 (e4m3) keys a tile, 64 a round of the four waves; tables for
# 4096 tokens let few pairs split up to 32 times, 168 pairs and more don't
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(
    "lens,Hkv,G,BS,most",
    [
        ([1, 15, 16, 17, 31, 32, 33], 2, 4, 64, 4096),
        ([63, 64, 65, 127, 129, 257, 1000], 1, 8, 16, 4096),
        ([2047, 2049, 1, 4000], 2, 7, 64, 4096),
        ([5, 100, 47], 3, 1, 8, None),     # pages smaller than a tile
        ([5, 100, 49, 97], 2, 5, 24, 4096),  # pages that cut tiles
        ([1, 33, 64, 80, 200, 17] * 4, 8, 3, 48, None),  # 192 pairs: one span
    ],
)
def test_attention_decode_edges(lens, Hkv, G, BS, most, fp8):
    kv, scales, wide, tables = _pages(lens, Hkv, BS, fp8, sum(lens) + G, most)
    B, Hq = len(lens), Hkv * G
    # rows 4 elements apart from dense: neither aligned nor contiguous
    q = torch.randn(B, Hq * D + 4, device=DEV).bfloat16()[:, : Hq * D].view(B, Hq, D)
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    got = ops.attention_decode(q, *kv, tables, ctx, k_scale=scales[0], v_scale=scales[1])
    dense = ops.attention_decode(q.contiguous(), *kv, tables, ctx, k_scale=scales[0],
                                 v_scale=scales[1])
    assert torch.equal(got, dense)
    for b, L in enumerate(lens):
        rows = tables[b, : -(-L // BS)].long()
        k, v = (x[rows].transpose(0, 1).reshape(Hkv, -1, D)[:, :L] for x in wide)
        ref = torch.cat([
            _softmax_rows(q[b, h * G:(h + 1) * G].double(), k[h], v[h]) for h in range(Hkv)
        ])
        # half a unit of bf16; fp32 sums of 128 products in the scores and
        # weights of 17 bits: 1e-4 of values of size 1
        torch.testing.assert_close(got[b].double(), ref, rtol=2**-8, atol=1e-4)


# an infinite value stays one, at the last key (whose row fills up its tile) and
# elsewhere, with one sign and both; a NaN, too
@pytest.mark.parametrize("B,most", [(3, 4096), (60, None)])
@pytest.mark.parametrize("at", [0, 33, 99])
def test_attention_decode_infinite_values(B, most, at):
    kv, _, _, tables = _pages([100] * B, 4, 16, False, B, most)
    v, dims = kv[1], {3: math.inf, 60: -math.inf, 101: math.nan}
    for d, x in dims.items():
        v[tables[1, at // 16], 2, at % 16, d] = x
    v[tables[1, 1], 2, 5, 7], v[tables[1, 4], 2, 5, 7] = math.inf, -math.inf
    q = torch.randn(B, 8, D, device=DEV).bfloat16() * 0.1
    ctx = torch.full((B,), 100, dtype=torch.int32, device=DEV)
    got = ops.attention_decode(q, *kv, tables, ctx)
    rows = got[1, 4:6]
    assert bool((rows[:, 3] == math.inf).all()) and bool((rows[:, 60] == -math.inf).all())
    assert bool(rows[:, [7, 101]].isnan().all())
    assert int((~got.isfinite()).sum()) == 8
    # scores that are not numbers leave none
    kv[0][tables[1, 0], 2, 1, 9] = math.nan
    assert bool(ops.attention_decode(q, *kv, tables, ctx)[1, 4:6].isnan().all())


# pages that the context before or behind has too are read another way than
# others: the same values come out
@pytest.mark.parametrize("fp8", [False, True])
def test_attention_decode_shared_pages(fp8):
    lens = [70, 300, 300, 200, 1, 300]
    kv, scales, _, tables = _pages(lens, 2, 16, fp8, 7, None)
    tables[2] = tables[1]  # as the one before, as the one behind; 0, 3, 4, 5 alone
    q = torch.randn(len(lens), 8, D, device=DEV).bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    got = ops.attention_decode(q, *kv, tables, ctx, k_scale=scales[0], v_scale=scales[1])
    at = torch.tensor([1, 0, 5, 2, 4, 3], device=DEV)  # no two neighbours alike
    apart = ops.attention_decode(
        q[at], *kv, tables[at], ctx[at], k_scale=scales[0], v_scale=scales[1])
    assert torch.equal(got[at], apart)


# 64 query rows and 64 keys a tile (32 keys with one head a kv head), 32 rows a
# wave, up to four heads a workgroup; pages in front of the step's own rows
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(
    "lens,cached,Hkv,G,BS",
    [
        ([1, 31, 32, 33, 64, 65, 129], 0, 2, 4, 64),
        ([1, 63, 100, 200], 1, 1, 1, 16),
        ([5, 64, 97], 31, 3, 1, 8),
        ([65, 2], 64, 2, 2, 24),
        ([1, 70, 33], 65, 2, 3, 64),
        ([40, 130], 129, 1, 5, 16),
        ([66], 63, 2, 6, 48),
        ([300, 1], 200, 2, 7, 64),
        ([90], 500, 1, 8, 64),
    ],
)
def test_attention_prefill_edges(lens, cached, Hkv, G, BS, fp8):
    if fp8 and not cached:
        pytest.skip("no pages, no bytes")
    B, Hq, T = len(lens), Hkv * G, sum(lens)
    torch.manual_seed(T + cached + G)
    # rows 4 elements apart from dense: neither aligned nor contiguous
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D + 4, device=DEV).bfloat16()
    q, k, v = (
        x.view(T, -1, D)
        for x in qkv[:, : (Hq + 2 * Hkv) * D].split([Hq * D, Hkv * D, Hkv * D], -1)
    )
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    cu_t = torch.tensor(cu, dtype=torch.int32, device=DEV)
    more = {}
    if cached:
        kv, scales, wide, tables = _pages([cached] * B, Hkv, BS, fp8, T)
        more = dict(
            k_cache=kv[0], v_cache=kv[1], block_tables=tables, k_scale=scales[0],
            v_scale=scales[1],
            cached_lens=torch.full((B,), cached, dtype=torch.int32, device=DEV),
        )
    got = ops.attention_prefill(q, k, v, cu_t, max(lens), **more)
    dense = ops.attention_prefill(
        q.contiguous(), k.contiguous(), v.contiguous(), cu_t, max(lens), **more
    )
    assert torch.equal(got, dense)
    for i, n in enumerate(lens):
        at = slice(cu[i], cu[i + 1])
        ks, vs = k[at].transpose(0, 1).double(), v[at].transpose(0, 1).double()
        if cached:
            rows = tables[i, : -(-cached // BS)].long()
            pages = (x[rows].transpose(0, 1).reshape(Hkv, -1, D)[:, :cached] for x in wide)
            ks, vs = (torch.cat([a, b], 1) for a, b in zip(pages, (ks, vs)))
        ahead = torch.ones(n, cached + n, dtype=torch.bool, device=DEV).triu(cached + 1)
        # weights are rounded to bf16, so sums of values are off by up to 2^-9 of
        # the largest; keys and values from bytes are rounded, too
        atol = float(vs.abs().max()) * (2**-7 if fp8 else 2**-9)
        for h in range(Hq):
            s = q[at, h].double() @ ks[h // G].T / math.sqrt(D)
            ref = s.masked_fill(ahead, -math.inf).softmax(-1) @ vs[h // G]
            torch.testing.assert_close(got[at, h].double(), ref, rtol=2**-8, atol=atol)


def _prompt_attention_in_order(q, k, v, cached):
    """[n, D] of one head over keys [cached + n, D]: 64 keys at a time (the cached
    ones apart), scores in fp32 relative to the largest so far, weights in bf16
    for the values and in fp32 for their sum."""
    n = q.shape[0]
    m = torch.full((n, 1), -math.inf, device=DEV)
    l = torch.zeros(n, 1, device=DEV)
    acc = torch.zeros(n, D, dtype=torch.float64, device=DEV)
    row = torch.arange(n, device=DEV).unsqueeze(1)
    for at in (*range(0, cached, 64), *range(cached, cached + n, 64)):
        end = min(at + 64, cached if at < cached else cached + n)
        s = (q.double() @ k[at:end].double().T).float() * torch.tensor(D**-0.5, device=DEV)
        s = s.masked_fill(torch.arange(at, end, device=DEV) > row + cached, -math.inf)
        top = torch.maximum(m, s.amax(-1, keepdim=True))
        w, factor = (s - top).exp(), (m - top).exp()
        l = l * factor + w.sum(-1, keepdim=True)
        acc = acc * factor.double() + w.bfloat16().double() @ v[at:end].double()
        m = top
    return (acc / l.double()).bfloat16()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(
    "n,cached,Hkv,G",
    [(37, 0, 2, 4), (300, 0, 2, 4), (130, 0, 4, 1), (200, 500, 2, 7), (257, 129, 1, 5),
     (700, 64, 8, 4), (65, 31, 1, 6)],
)
def test_attention_prefill_order(n, cached, Hkv, G, fp8):
    """However heads are shared out, sums are in the order above: but for the last
    bit of fp32 sums, which shows in few roundings to bf16, the same comes out."""
    if fp8 and not cached:
        pytest.skip("no pages, no bytes")
    torch.manual_seed(n + cached)
    q, k, v = ((torch.randn(n, h, D, device=DEV) * 1.3).bfloat16() for h in (Hkv * G, Hkv, Hkv))
    more, keys = {}, [k.transpose(0, 1), v.transpose(0, 1)]
    if cached:
        kv, scales, wide, tables = _pages([cached], Hkv, 64, fp8, n)
        more = dict(
            k_cache=kv[0], v_cache=kv[1], block_tables=tables,
            cached_lens=torch.tensor([cached], dtype=torch.int32, device=DEV),
            k_scale=scales[0], v_scale=scales[1],
        )
        pages = (x[tables[0].long()].transpose(0, 1).reshape(Hkv, -1, D)[:, :cached] for x in wide)
        keys = [torch.cat([a.float().bfloat16(), b], 1) for a, b in zip(pages, keys)]
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    got = ops.attention_prefill(q, k, v, cu, n, **more)
    want = torch.stack([
        _prompt_attention_in_order(q[:, h], keys[0][h // G], keys[1][h // G], cached)
        for h in range(Hkv * G)
    ], 1)
    # fp32 sums and exponentials are off by some 2^-22, so of the weights, 2^-8 of
    # themselves apart, one in 2^13 rounds to its neighbour: a result changes by
    # 2^-8 of one weight in thousands, or 2^-22 by its own sum, and rounds to its
    # neighbour in a percent of cases. Weights that are relative to anything but
    # the largest so far turn a fifth and more.
    differ = float((got != want).double().mean())
    assert differ < 0.02, differ


# behind the last key a tile has its row again, with weights of 0
@pytest.mark.parametrize("cached", [0, 70])
def test_attention_prefill_infinite_values(cached):
    torch.manual_seed(5)
    n, Hkv, G = 70, 2, 2
    q, k, v = (torch.randn(n, h, D, device=DEV).bfloat16() for h in (Hkv * G, Hkv, Hkv))
    more = {}
    if cached:
        kv, _, _, tables = _pages([cached], Hkv, 64, False, 3)
        kv[1][tables[0, 1], 1, 5, 7] = -math.inf  # the last one
        more = dict(
            k_cache=kv[0], v_cache=kv[1], block_tables=tables,
            cached_lens=torch.tensor([cached], dtype=torch.int32, device=DEV),
        )
    else:
        v[-1, 1, 7] = -math.inf
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    got = ops.attention_prefill(q, k, v, cu, n, **more)
    sees = slice(None) if cached else slice(n - 1, None)
    assert bool((got[sees, G:, 7] == -math.inf).all())
    assert bool(got[:, :G].isfinite().all()) and bool(got[:64].isfinite().all() or cached)


# rows that start off 16 bytes (odd V), shorter than the workgroup, more equal
# tokens than the list of a coarse bin holds, masked and NaN tokens
@pytest.mark.parametrize("V", [5, 63, 1000, 4097, 32003, 128256])
def test_topk_topp_filter_rows(V):
    g = torch.Generator(device=DEV).manual_seed(V)
    x = torch.randn(9, V, generator=g, device=DEV) * 2.5
    x[1, : V // 2] = -math.inf
    x[2] = 1.0                   # all tie: a cut keeps all
    x[3] = x[3].clamp(max=0.5)   # half of the row ties at the top
    x[4, V // 3] = 40.0          # one token has all the mass
    x[5, 0] = math.nan
    topp = torch.tensor([0.9, 0.95, 0.5, 1.0, 0.9, 0.9, 0.0, 1.0, 1.0], device=DEV)
    topk = torch.tensor([0, 20, 3, 7, 0, 0, 0, V, 0], dtype=torch.int32, device=DEV)
    got = ops.topk_topp_filter(x.clone(), topp, topk)
    assert torch.equal(got[8], x[8]) and torch.equal(got[7], x[7])
    assert torch.equal(got[5].isnan(), x[5].isnan())  # no mass is enough there
    assert torch.equal(got[5][1:], x[5][1:])
    for b in (0, 1, 2, 3, 4, 6):
        ranked = x[b].double().sort(descending=True).values
        p = ranked.softmax(-1)
        keep = (p.cumsum(-1) - p < topp[b].double()) | (topp[b] >= 1)
        if topk[b] > 0:
            keep &= torch.arange(V, device=DEV) < topk[b]
        least = ranked[int(keep.sum()) - 1] if bool(keep.any()) else ranked[0]
        kept = got[b] > -math.inf
        # what lies within the cut's granularity (16/2048^2) of it stays, too;
        # masses are multiples of 2^-42 and exponentials good to 2^-22, so a
        # token may change sides where the mass in front of it is that close
        sure = x[b].double() >= least
        near = x[b].double() >= least - 4e-6
        extra = (kept & ~near).sum() + (sure & ~kept).sum()
        assert int(extra) <= (1 if topp[b] < 1 else 0), (V, b, int(extra))
        assert torch.equal(got[b][kept], x[b][kept])


# many tokens of next to no mass, which together reach into what is asked for:
# each is far below 2^-31 of the largest
@pytest.mark.parametrize("V", [32000, 90000, 128256])
@pytest.mark.parametrize("B", [1, 3, 70])
def test_filter_counts_small_masses(V, B):
    x = torch.full((B, V), -22.5, device=DEV)
    x[:, V // 2] = 0.0
    tail = math.exp(-22.5) * (V - 1)
    topk = torch.zeros(B, dtype=torch.int32, device=DEV)
    # the first token alone is enough up to 1 / (1 + tail), 4e-6 to 2e-5 below 1
    for p, kept in ((1 - 1.5 * tail, 1), (1 - 0.5 * tail, V)):
        got = ops.topk_topp_filter(x.clone(), torch.full((B,), p, device=DEV), topk)
        assert ((got > -math.inf).sum(1) == kept).all(), (p, kept)


# rows in 16, 5 and 4 pieces and whole ones: the same tokens stay
@pytest.mark.parametrize("V", [98304, 98307, 128256, 152066])
def test_filter_pieces(V):
    g = torch.Generator(device=DEV).manual_seed(V)
    x = torch.randn(11, V, generator=g, device=DEV) * 2.5
    x[1, : V // 2] = -math.inf
    x[2] = 1.0                    # more of a bin than its list holds
    x[3] = x[3].clamp(max=0.5)
    x[4, V // 3] = 40.0
    x[5, 0] = math.nan
    x[6] = -math.inf
    x[7, V - 1] = math.inf
    topp = torch.tensor([0.9, 0.95, 0.5, 1.0, 0.9, 0.9, 0.9, 0.5, 1.0, 1.0, 0.3], device=DEV)
    topk = torch.tensor([0, 20, 3, 7, 0, 0, 5, 0, V, 0, 1], dtype=torch.int32, device=DEV)
    whole = ops.topk_topp_filter(x.repeat(24, 1), topp.repeat(24), topk.repeat(24))[:11]
    for b in range(11):
        alone = ops.topk_topp_filter(x[b : b + 1].clone(), topp[b : b + 1], topk[b : b + 1])
        assert torch.equal(alone.view(torch.int32), whole[b : b + 1].view(torch.int32)), b
    for times in (1, 4, 5, 6):
        rows = ops.topk_topp_filter(x.repeat(times, 1), topp.repeat(times), topk.repeat(times))
        for part in rows.split(11):
            assert torch.equal(part.view(torch.int32), whole.view(torch.int32)), times


@pytest.mark.parametrize("V", [3, 64, 4095, 4096, 32000, 128257])
def test_sample_rows(V):
    g = torch.Generator(device=DEV).manual_seed(V)
    x = torch.randn(6, V, generator=g, device=DEV) * 2
    x[1, V // 2:] = -math.inf
    x[2] = -math.inf
    temps = torch.tensor([0.7, 1.0, 0.5, 0.0, 1.3, 0.9], device=DEV)
    noise = torch.rand(6, V, generator=g, device=DEV)
    got = ops.sample(x, temps, noise)
    u = noise.double().clamp_min(1e-20)
    score = x.double() / temps.double().clamp_min(1e-6).unsqueeze(1) - (-u.log()).clamp_min(1e-20).log()
    score[3] = x[3].double()
    assert int(got[2]) == 0  # all masked: the first
    for b in (0, 1, 3, 4, 5):
        # fp32 logarithms and sums of numbers below 32: 1e-5
        assert float(score[b, got[b]]) >= float(score[b].max()) - 1e-5


# 16 rows and columns a block, depth in tiles of 64 and 128 shared by up to 8
# waves: remainders of rows, of the last tile, fewer tiles than waves
@pytest.mark.parametrize("M", [1, 3, 16, 17, 32, 33, 47, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(64, 32), (64, 160), (192, 1056), (4160, 512), (4096, 96)])
def test_gemm_stream_edges(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
    ref = x.double() @ w.double().T
    # half a unit of bf16, and fp32 sums of K products of size 1/sqrt(K)
    atol = 2**-24 * K * float(x.abs().max()) * float(w.abs().max())
    for swiglu in (False, True):
        if M > 48 and swiglu:
            continue
        rows = torch.full((M + 2, N // 2 if swiglu else N), 7.0, device=DEV).bfloat16()
        ops._shared().gemm_stream(rows[1:-1], x, w, swiglu)
        assert bool((rows[0] == 7).all()) and bool((rows[-1] == 7).all())
        want = ref
        if swiglu:
            gate, up = ref.chunk(2, -1)
            want = torch.nn.functional.silu(gate) * up
        # both sums' errors, times the other's size, and of an exponential
        scale = 2 * float(ref.abs().max()) + 1 if swiglu else 1
        torch.testing.assert_close(
            rows[1:-1].double(), want, rtol=2**-8, atol=atol * scale + (1e-5 if swiglu else 0))


def test_gemm_stream_refuses():
    x = torch.zeros(65, 64, device=DEV).bfloat16()
    w = torch.zeros(64, 64, device=DEV).bfloat16()
    y = torch.zeros(65, 64, device=DEV).bfloat16()
    with pytest.raises(RuntimeError):
        ops._shared().gemm_stream(y, x, w, False)
    off = torch.zeros(64 * 64 + 1, device=DEV).bfloat16()[1:].view(64, 64)
    with pytest.raises(RuntimeError):  # not aligned
        ops._shared().gemm_stream(y[:4], x[:4], off, False)
    # what it does not take still runs
    assert ops.linear(x[:4], off).shape == (4, 64)


def test_linear_of_other_operands():
    """What gemm_stream does not take goes where it went: products to be derived,
    without columns or depth."""
    x = torch.randn(32, 64, device=DEV).bfloat16()
    w = torch.randn(128, 64, device=DEV).bfloat16()
    for a, b in ((x.clone().requires_grad_(), w), (x, w.clone().requires_grad_())):
        ops.linear(a, b).float().sum().backward()
        wide = [t.detach().float().requires_grad_(t.requires_grad) for t in (a, b)]
        torch.nn.functional.linear(*wide).sum().backward()
        for t, u in zip((a, b), wide):
            if t.requires_grad:
                torch.testing.assert_close(t.grad.float(), u.grad, rtol=2**-7, atol=2**-5)
    with torch.no_grad():
        got = ops.linear(x.clone().requires_grad_(), w)
    assert torch.equal(got, ops.linear(x, w))
    assert ops.linear(x, w[:0]).shape == (32, 0)
    assert bool((ops.linear(x[:, :0], w[:, :0]) == 0).all())


# a block of 16 rows and two, tiles that end inside a row, few and many column
# blocks; against float64 from the same bf16 stream
@pytest.mark.parametrize("T", [1, 5, 16, 17, 32])
@pytest.mark.parametrize("H,Hq,Hkv,I", [(256, 2, 1, 128), (1056, 4, 2, 4160), (4096, 32, 8, 512)])
def test_streamed_layer(T, H, Hq, Hkv, I):
    g = torch.Generator(device=DEV).manual_seed(T + H)

    def rand(*shape, by=1.0):
        return (torch.randn(*shape, generator=g, device=DEV) * by).bfloat16()

    r, norm = rand(T, H, by=3.0), rand(H)
    eps, BS, NB = 1e-5, 16, 9
    wide = r.double()
    normed = wide * torch.rsqrt(wide.square().mean(-1, keepdim=True) + eps) * norm.double()

    w = rand((Hq + 2 * Hkv) * D, H, by=H**-0.5)
    cs = ops.build_rope_cache(600, D, 10000.0, device=DEV)
    positions = torch.randint(0, 600, (T,), generator=g, device=DEV)
    slots = torch.randperm(NB * BS, generator=g, device=DEV)[:T]
    slots[0] = -1
    caches = [torch.full((NB, Hkv, BS, D), 7.0, device=DEV).bfloat16() for _ in range(2)]
    got = ops.norm_qkv_rotated(r, norm, eps, w, positions, cs, slots, *caches)
    heads = (normed @ w.double().T).view(T, -1, D)
    cos, sin = (x[:, None] for x in cs[positions].double().split(D // 2, -1))
    a, b = heads[:, : Hq + Hkv].split(D // 2, -1)
    want = torch.cat([torch.cat([a * cos - b * sin, b * cos + a * sin], -1), heads[:, Hq + Hkv:]], 1)
    # the normed row is rounded to 2^-9, H products of size 1/sqrt(H): 4 of
    # their sums' deviations; the output to 2^-9
    near = dict(rtol=2**-8, atol=4 * 2**-9 * float(norm.double().abs().max()))
    torch.testing.assert_close(got.view(T, -1, D).double(), want, **near)
    for cache, first in zip(caches, (Hq, Hq + Hkv)):
        expect = torch.full_like(cache, 7.0)
        at = slots[1:]
        expect[at // BS, :, at % BS] = got.view(T, -1, D)[1:, first:first + Hkv]
        assert torch.equal(cache, expect)

    w = rand(2 * I, H, by=H**-0.5)
    got = ops.norm_swiglu_linear(r, norm, eps, w)
    gate, up = (normed @ w.double().T).chunk(2, -1)
    big = float(torch.maximum(gate.abs().max(), up.abs().max()))
    torch.testing.assert_close(
        got.double(), torch.nn.functional.silu(gate) * up, rtol=2**-8, atol=2 * big * near["atol"])

    x, w = rand(T, I), rand(H, I, by=I**-0.5)
    got = ops.linear_add_(x, w, r.clone())
    torch.testing.assert_close(
        got.double(), wide + x.double() @ w.double().T, rtol=2**-8, atol=2**-24 * I)

    if T <= 16:
        w = rand(512, H, by=H**-0.5)
        got = ops.norm_logits(r, norm, eps, w)
        assert got.dtype == torch.float32
        torch.testing.assert_close(got.double(), normed @ w.double().T, **near)


# queries, keys and values of more than 8192 columns, additions to more than 4096:
# workgroups of four waves
@pytest.mark.parametrize("T", [1, 5, 16, 17, 32])
@pytest.mark.parametrize("H,Hq,Hkv,I", [(4160, 56, 8, 256), (5120, 64, 2, 1024), (8192, 64, 8, 160)])
def test_streamed_layer_wide(T, H, Hq, Hkv, I):
    test_streamed_layer(T, H, Hq, Hkv, I)


# what gemm_stream does not take of few rows: rows that end inside a tile, one
# slab of K and several, operands that start anywhere
@pytest.mark.parametrize("M", [1, 3, 15, 16])
@pytest.mark.parametrize("N,K", [(64, 32), (192, 1056), (4096, 4096), (1024, 14336)])
def test_gemm_skinny_rows(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    x = torch.randn(M * K + 1, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N * K + 1, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
    # half a unit of bf16, and fp32 sums of K products of size 1/sqrt(K)
    near = dict(rtol=2**-8, atol=2**-24 * K * float(x.abs().max()) * float(w.abs().max()))
    for off in (0, 1):
        a, b = x[off:][: M * K].view(M, K), w[off:][: N * K].view(N, K)
        ref = a.double() @ b.double().T
        nsk = ops._skinny_nsk(N, K)
        assert nsk > 1 or K < 4096
        ws = ops._skinny_scratch(x.device, nsk * M * N) if nsk > 1 else None
        rows = torch.full((M + 2, N), 7.0, device=DEV).bfloat16()
        ops._shared().gemm_skinny(rows[1:-1], a, b, ws, nsk, False)
        torch.testing.assert_close(rows[1:-1].double(), ref, **near)
        assert bool((rows[0] == 7).all()) and bool((rows[-1] == 7).all())
        torch.testing.assert_close(ops.linear(a, b).double(), ref, **near)
    assert not ops._streamable(a, b)


def test_streamed_steps_match_others():
    """A step whose layers go to gemm_stream and the same step by separate
    kernels (a row more than they take, padded) agree to bf16's rounding."""
    from llmapigateway_amd.engine.kvcache import PagedKVCache
    from llmapigateway_amd.models import build_model
    from llmapigateway_amd.models.batch import ForwardBatch
    from llmapigateway_amd.models.configs import ModelConfig

    c = ModelConfig(
        name="few-rows", hidden_size=512, intermediate_size=1024, num_layers=2, num_heads=4,
        num_kv_heads=2, vocab_size=2048, head_dim=128, rope_theta=10000.0, max_positions=1024,
    )
    model = build_model(c, device=DEV, dtype=torch.bfloat16, seed=3)
    assert ops.layer_streams(32, model.layers[0]) and not ops.layer_streams(33, model.layers[0])
    logits = []
    for T in (32, 33):
        cache = PagedKVCache(c, 40, 16, DEV, torch.bfloat16)
        n = torch.arange(T, device=DEV)
        batch = ForwardBatch(
            kind="decode", token_ids=n * 7 % 2048, positions=n % 16, slot_mapping=n * 16 + n % 16,
            block_tables=n.int().unsqueeze(1).contiguous(), context_lens=(n % 16 + 1).int(),
        )
        for k in cache.k_caches + cache.v_caches:
            k.copy_(torch.linspace(-1, 1, k.numel(), device=DEV).view(k.shape))
        logits.append(model.step(batch, cache)[:32])
    # two layers, each of whose ten roundings is 2^-9
    diff = (logits[0] - logits[1]).norm() / logits[1].norm()
    assert float(diff) < 0.02, float(diff)


@pytest.mark.parametrize("T", [4, 40])
def test_fused_swiglu_switch(T, monkeypatch):
    """LLMAPI_NO_FUSED_SWIGLU takes swiglu apart from its product, of few rows and
    of tiles, and leaves the rest of the layer as it is."""
    from llmapigateway_amd.engine.kvcache import PagedKVCache
    from llmapigateway_amd.models import build_model
    from llmapigateway_amd.models.batch import ForwardBatch
    from llmapigateway_amd.models.configs import ModelConfig

    c = ModelConfig(
        name="rows", hidden_size=2048, intermediate_size=1024, num_layers=2, num_heads=4,
        num_kv_heads=2, vocab_size=2048, head_dim=128, rope_theta=10000.0, max_positions=1024,
    )
    model = build_model(c, device=DEV, dtype=torch.bfloat16, seed=3)
    n = torch.arange(T, device=DEV)
    apart, calls = ops.swiglu, []
    monkeypatch.setattr(ops, "swiglu", lambda x: calls.append(x.shape) or apart(x))
    routes, logits = [], []
    for switch in ("", "1"):
        monkeypatch.setenv("LLMAPI_NO_FUSED_SWIGLU", switch)
        first = model.layers[0]
        routes.append((ops.layer_streams(T, first), ops.layer_tiles(T, first, 128)))
        cache = PagedKVCache(c, 40, 16, DEV, torch.bfloat16)
        logits.append(model.step(ForwardBatch(
            kind="decode", token_ids=n, positions=n % 16, slot_mapping=n * 16 + n % 16,
            block_tables=n.int().unsqueeze(1).contiguous(), context_lens=(n % 16 + 1).int(),
        ), cache))
        assert len(calls) == (2 if switch else 0)
    assert routes[0] == routes[1] and any(routes[0])
    diff = (logits[0] - logits[1]).norm() / logits[0].norm()
    assert float(diff) < 0.02, float(diff)  # two layers, each of whose ten roundings is 2^-9


@pytest.mark.parametrize("H", [4, 12, 16392])
def test_embed_rows_of_other_sizes(H):
    """What the kernel does not hold is gathered."""
    embed = torch.randn(70, H, device=DEV).bfloat16()
    tokens = torch.randint(0, 70, (9,), device=DEV)
    r, x = ops.embed_rows(tokens, embed, torch.ones(H, device=DEV).bfloat16(), 1e-5, normed=False)
    assert x is None and torch.equal(r, embed[tokens])


@pytest.mark.parametrize("T", [4, 40])
def test_norm_weights_off_16_bytes(T):
    """Layers whose norms' weights are views that start anywhere, by few rows and
    tiles: as with weights that lie alone."""
    from llmapigateway_amd.engine.kvcache import PagedKVCache
    from llmapigateway_amd.models import build_model
    from llmapigateway_amd.models.batch import ForwardBatch
    from llmapigateway_amd.models.configs import ModelConfig

    c = ModelConfig(
        name="rows", hidden_size=2048, intermediate_size=1024, num_layers=2, num_heads=4,
        num_kv_heads=2, vocab_size=2048, head_dim=128, rope_theta=10000.0, max_positions=1024,
    )
    model = build_model(c, device=DEV, dtype=torch.bfloat16, seed=3)

    def off(w):
        return torch.cat([w.new_zeros(1), w])[1:]

    n = torch.arange(T, device=DEV)
    logits = []
    for kv in ("auto", "fp8"):
        for _ in range(2):
            cache = PagedKVCache(c, 40, 16, DEV, torch.bfloat16, kv_dtype=kv)
            logits.append(model.step(ForwardBatch(
                kind="decode", token_ids=n, positions=n % 16, slot_mapping=n * 16 + n % 16,
                block_tables=n.int().unsqueeze(1).contiguous(), context_lens=(n % 16 + 1).int(),
            ), cache))
            for layer in model.layers:
                layer.update({k: off(layer[k]) for k in ("input_norm", "post_norm")})
            model.final_norm = off(model.final_norm)
        assert torch.equal(*logits[-2:])


@pytest.mark.parametrize("T", [4, 40, 600])
def test_steps_without_logits(T):
    """A step that asks for no row's logits gets none, by few rows, tiles and
    separate kernels."""
    from llmapigateway_amd.engine.kvcache import PagedKVCache
    from llmapigateway_amd.models import build_model
    from llmapigateway_amd.models.batch import ForwardBatch
    from llmapigateway_amd.models.configs import ModelConfig

    c = ModelConfig(
        name="rows", hidden_size=2048, intermediate_size=1024, num_layers=1, num_heads=4,
        num_kv_heads=2, vocab_size=2048, head_dim=128, rope_theta=10000.0, max_positions=1024,
    )
    model = build_model(c, device=DEV, dtype=torch.bfloat16, seed=3)
    cache = PagedKVCache(c, 40, 16, DEV, torch.bfloat16)
    n = torch.arange(T, device=DEV)
    tile_seq, tile_off = ops.build_prefill_tiles([T], torch.device(DEV))
    batch = ForwardBatch(
        kind="prefill", token_ids=n, positions=n, slot_mapping=n,
        cu_seqlens=torch.tensor([0, T], dtype=torch.int32, device=DEV), max_seqlen=T,
        tile_seq=tile_seq, tile_off=tile_off,
        logits_indices=torch.zeros(0, dtype=torch.long, device=DEV),
    )
    got = model.step(batch, cache)
    assert got.shape == (0, 2048) and got.dtype == torch.float32
    # the rows are in their pages all the same
    pages = cache.k_caches[0].transpose(1, 2).reshape(-1, 2 * D)
    assert bool((pages[:T] != 0).any(1).all()) and bool((pages[T:] == 0).all())


# tiles of 64, 128 and 256 rows, of 64 to 256 columns; one tile of depth and
# more splits than there are; columns and rows that end inside a tile
@pytest.mark.parametrize("M", [1, 17, 64, 65, 128, 129, 200, 256, 257, 385, 512])
@pytest.mark.parametrize(
    "N,K", [(32, 64), (96, 192), (4096, 512), (4640, 576), (160, 8256), (33088, 128), (50080, 64)])
def test_gemm_tile_edges(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
    ref = x.double() @ w.double().T
    # fp32 sums of K products
    atol = 2**-24 * K * float(x.abs().max()) * float(w.abs().max())
    splits = ops._native().gemm_tile_splits(M, N, K)
    for y in (
        torch.full((splits, M, N), 7.0, device=DEV), torch.full((3, M, N), 7.0, device=DEV),
        torch.full((M, N), 7.0, device=DEV),
        torch.full((M, N // 2), 7.0, device=DEV, dtype=torch.bfloat16),
    ):
        if M > 256 and y.dim() == 2:
            continue
        rows = torch.cat([y.flatten(), y.new_full((64,), 7.0)])  # and what lies behind
        ops._native().gemm_tile(rows[:-64].view(y.shape), x, w)
        assert bool((rows[-64:] == 7).all())
        got, want, scale, rtol = rows[:-64].view(y.shape).double(), ref, 1, 0
        if y.dim() == 3:
            got = got.sum(0)
        elif y.dtype == torch.bfloat16:
            gate, up = ref.chunk(2, -1)
            want = torch.nn.functional.silu(gate) * up
            scale, rtol = 2 * float(ref.abs().max()) + 1, 2**-8
        torch.testing.assert_close(got, want, rtol=rtol, atol=atol * scale + (1e-5 if rtol else 0))


# 16385 to 32768 columns: tiles of 128 of them
@pytest.mark.parametrize("M", [1, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("N,K", [(16416, 192), (28704, 64), (32768, 320)])
def test_gemm_tile_wide(M, N, K):
    test_gemm_tile_edges(M, N, K)


def test_gemm_tile_refuses():
    def call(M, N, K, y, off=0):
        x = torch.zeros(M * K + off, device=DEV).bfloat16()[off:].view(M, K)
        ops._native().gemm_tile(y, x, torch.zeros(N, K, device=DEV).bfloat16())

    fp32 = dict(device=DEV, dtype=torch.float32)
    for args in (
        (257, 64, 64, torch.zeros(257, 64, **fp32)), (513, 64, 64, torch.zeros(2, 513, 64, **fp32)),
        (4, 24, 64, torch.zeros(4, 24, **fp32)),
        (4, 64, 32, torch.zeros(4, 64, **fp32)), (4, 64, 64, torch.zeros(4, 32, **fp32)),
        (4, 48, 64, torch.zeros(4, 24, device=DEV).bfloat16()),
        (4, 64, 64, torch.zeros(4, 64, **fp32), 4),
    ):
        with pytest.raises(RuntimeError):
            call(*args)


@pytest.mark.parametrize("T,splits", [(2, 1), (33, 3), (200, 8), (5, 9)])
@pytest.mark.parametrize("H,Hq,Hkv", [(8, 1, 1), (2056, 4, 1), (3584, 28, 4), (16384, 5, 5)])
def test_parts_rows(T, splits, H, Hq, Hkv):
    g = torch.Generator(device=DEV).manual_seed(T + H)
    r = (torch.randn(T, H, generator=g, device=DEV) * 3).bfloat16()
    norm = torch.randn(H, generator=g, device=DEV).bfloat16()
    parts = torch.randn(splits, T, H, generator=g, device=DEV)
    total = r.double() + parts.double().sum(0)
    x = ops.add_parts_norm_(r, parts, norm, 1e-5)
    # a half unit of bf16, and splits fp32 additions of numbers below 64
    torch.testing.assert_close(r.double(), total, rtol=2**-8, atol=2**-18 * splits)
    wide = r.double()
    want = wide * torch.rsqrt(wide.square().mean(-1, keepdim=True) + 1e-5) * norm.double()
    torch.testing.assert_close(x.double(), want, rtol=2**-8 + 2**-18, atol=1e-6)

    BS, NB, N = 16, 14, (Hq + 2 * Hkv) * D
    parts = torch.randn(splits, T, N, generator=g, device=DEV)
    cs = ops.build_rope_cache(600, D, 10000.0, device=DEV)
    positions = torch.randint(0, 600, (T,), generator=g, device=DEV)
    slots = torch.randperm(NB * BS, generator=g, device=DEV)[:T]
    slots[T // 2] = -1
    heads = parts.double().sum(0).view(T, -1, D)
    cos, sin = (x[:, None] for x in cs[positions].double().split(D // 2, -1))
    a, b = heads[:, : Hq + Hkv].split(D // 2, -1)
    want = torch.cat([torch.cat([a * cos - b * sin, b * cos + a * sin], -1), heads[:, Hq + Hkv:]], 1)
    kept = torch.arange(T, device=DEV) != T // 2
    for fp8 in (False, True):
        caches = [
            torch.full((NB, Hkv, BS, D), 7.0, device=DEV)
            .to(torch.uint8 if fp8 else torch.bfloat16) for _ in range(2)
        ]
        expect = [c.clone() for c in caches]
        scales = [torch.zeros(NB, Hkv, BS, device=DEV) for _ in range(2)] if fp8 else [None, None]
        again = [torch.zeros(NB, Hkv, BS, device=DEV) for _ in range(2)] if fp8 else [None, None]
        got = ops.rotated_parts(
            parts, positions, cs, slots, *caches, k_scale=scales[0], v_scale=scales[1])
        torch.testing.assert_close(
            got.view(T, -1, D).double(), want, rtol=2**-8, atol=2**-17 * splits)
        # the pages hold what the page writer makes of those rows
        _, k, v = got.view(T, -1, D)[kept].split([Hq, Hkv, Hkv], 1)
        ops.kv_cache_write(k, v, *expect, slots[kept], k_scale=again[0], v_scale=again[1])
        for one, other in zip(caches, expect):
            assert torch.equal(one, other)
        if fp8:
            assert torch.equal(scales[0], again[0]) and torch.equal(scales[1], again[1])


@pytest.mark.parametrize("T", [1, 300])
@pytest.mark.parametrize("H", [8, 1024, 1032, 3584, 8192, 16384])
def test_embed_rows(T, H):
    g = torch.Generator(device=DEV).manual_seed(T + H)
    embed = torch.randn(70, H, generator=g, device=DEV).bfloat16()
    w = torch.randn(H, generator=g, device=DEV).bfloat16()
    tokens = torch.randint(0, 70, (T,), generator=g, device=DEV)
    tokens[-1] = 69
    r, x = ops.embed_rows(tokens, embed, w, 1e-5)
    assert torch.equal(r, embed[tokens])
    wide = r.double()
    want = wide * torch.rsqrt(wide.square().mean(-1, keepdim=True) + 1e-5) * w.double()
    torch.testing.assert_close(x.double(), want, rtol=2**-8 + 2**-18, atol=1e-6)
    again, none = ops.embed_rows(tokens, embed, w, 1e-5, normed=False)
    assert none is None and torch.equal(again, r)


@pytest.mark.parametrize("H", [512, 4096])
def test_embed_rows_unknown_tokens(H):
    embed = torch.randn(70, H, device=DEV).bfloat16()
    w = torch.ones(H, device=DEV).bfloat16()
    tokens = torch.tensor([3, -1, 69, 70, 2**40], device=DEV)
    for normed in (False, True):
        r, x = ops.embed_rows(tokens, embed, w, 1e-5, normed=normed)
        assert torch.equal(r[::2][:2], embed[[3, 69]])
        for rows in (r, x) if normed else (r,):
            assert bool(rows[[1, 3, 4]].isnan().all()) and bool(rows[[0, 2]].isfinite().all())


@pytest.mark.parametrize("fp8", [False, True])
def test_tiled_steps_match_others(fp8, monkeypatch):
    """A step whose products go to gemm_tile (of 9 and 20 rows to gemm_stream) and the
    same step by separate kernels agree to bf16's rounding."""
    from llmapigateway_amd.engine.kvcache import PagedKVCache
    from llmapigateway_amd.models import build_model
    from llmapigateway_amd.models.batch import ForwardBatch
    from llmapigateway_amd.models.configs import ModelConfig

    c = ModelConfig(
        name="rows", hidden_size=2048, intermediate_size=1024, num_layers=2, num_heads=4,
        num_kv_heads=2, vocab_size=2048, head_dim=128, rope_theta=10000.0, max_positions=1024,
    )
    model = build_model(c, device=DEV, dtype=torch.bfloat16, seed=3)
    for T in (9, 17, 20, 40, 250, 300, 512):
        logits = []
        for separate in (False, True):
            if separate or T not in (9, 20):
                monkeypatch.setattr(ops, "layer_streams", lambda *a: False)
            if separate:
                monkeypatch.setattr(ops, "layer_tiles", lambda *a: False)
            first = model.layers[0]
            assert separate or ops.layer_streams(T, first) or ops.layer_tiles(T, first, 128)
            cache = PagedKVCache(c, 520, 16, DEV, torch.bfloat16, kv_dtype="fp8" if fp8 else "auto")
            n = torch.arange(T, device=DEV)
            batch = ForwardBatch(
                kind="decode", token_ids=n * 7 % 2048, positions=n % 16,
                slot_mapping=n * 16 + n % 16,
                block_tables=n.int().unsqueeze(1).contiguous(), context_lens=(n % 16 + 1).int(),
            )
            if fp8:
                for k in cache.k_scales + cache.v_scales:
                    k.fill_(0.01)
            else:
                for k in cache.k_caches + cache.v_caches:
                    k.copy_(torch.linspace(-1, 1, k.numel(), device=DEV).view(k.shape))
            logits.append(model.step(batch, cache))
        monkeypatch.undo()
        assert logits[0].dtype == torch.float32
        # two layers, each of whose ten roundings is 2^-9; a row in e4m3 2^-4
        diff = (logits[0] - logits[1]).norm() / logits[1].norm()
        assert float(diff) < (0.05 if fp8 else 0.02), float(diff)


def _steps_of(c, lens, cached, decodes, kv):
    """A mixed step (of prompts alone where decodes is 0) and pages for it."""
    from llmapigateway_amd.engine.kvcache import PagedKVCache
    from llmapigateway_amd.models.batch import ForwardBatch

    g = torch.Generator(device=DEV).manual_seed(sum(lens) + cached)
    B, BS = len(lens) + decodes, 16
    width = -(-(max(lens + [40]) + cached) // BS)
    cache = PagedKVCache(c, B * width, BS, DEV, torch.bfloat16, kv_dtype=kv)
    for pages, scale in zip(cache.k_caches + cache.v_caches,
                            (cache.k_scales + cache.v_scales) if cache.fp8 else [None] * 99):
        x = torch.randn(pages.shape, generator=g, device=DEV)
        if cache.fp8:
            pages.copy_((x * 64).to(torch.float8_e4m3fn).view(torch.uint8))
            scale.fill_(0.02)
        else:
            pages.copy_(x)
    tables = torch.randperm(B * width, generator=g, device=DEV).int().view(B, width)
    context = torch.arange(decodes, device=DEV) % 40 + 1
    positions = torch.cat(
        [torch.arange(cached, cached + n, device=DEV) for n in lens] + [context - 1])
    row = torch.tensor([i for i, n in enumerate(lens) for _ in range(n)], device=DEV)
    row = torch.cat([row, torch.arange(len(lens), B, device=DEV)])
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    tile_seq, tile_off = ops.build_prefill_tiles(lens, torch.device(DEV))
    more = {}
    if cached:
        more.update(block_tables=tables[: len(lens)].contiguous(),
                    cached_lens=torch.full((len(lens),), cached, dtype=torch.int32, device=DEV))
    if decodes:
        more.update(dec_block_tables=tables[len(lens):].contiguous(),
                    dec_context_lens=context.int())
    T = len(row)
    return cache, ForwardBatch(
        kind="mixed" if decodes else "prefill",
        token_ids=torch.randint(0, c.vocab_size, (T,), generator=g, device=DEV),
        positions=positions, slot_mapping=tables[row, positions // BS].long() * BS + positions % BS,
        cu_seqlens=cu, max_seqlen=max(lens), tile_seq=tile_seq, tile_off=tile_off,
        n_prefill_tokens=sum(lens),
        logits_indices=torch.cat([cu[1:].long() - 1, torch.arange(sum(lens), T, device=DEV)]),
        **more,
    )


@pytest.mark.parametrize("kv", ["auto", "fp8"])
@pytest.mark.parametrize(
    "lens,cached,decodes",
    [([7], 0, 0), ([5, 3], 33, 4), ([11], 0, 21), ([40, 9], 0, 0), ([70, 1], 20, 30),
     ([300], 0, 100), ([200, 57], 64, 3)],
)
def test_prompt_and_mixed_steps_match_others(lens, cached, decodes, kv, monkeypatch):
    """Steps over prompts, with and without decoded rows beside them, by few rows
    or tiles (e4m3: in order) and by separate kernels agree to bf16's rounding."""
    from llmapigateway_amd.models import build_model
    from llmapigateway_amd.models.configs import ModelConfig

    c = ModelConfig(
        name="rows", hidden_size=2048, intermediate_size=1024, num_layers=2, num_heads=4,
        num_kv_heads=2, vocab_size=2048, head_dim=128, rope_theta=10000.0, max_positions=1024,
    )
    model = build_model(c, device=DEV, dtype=torch.bfloat16, seed=3)
    got = []
    T = sum(lens) + decodes
    assert ops.layer_streams(T, model.layers[0]) or ops.layer_tiles(T, model.layers[0], 128)
    for separate in (False, True):
        if separate:
            for route in ("layer_streams", "layer_tiles", "_streamable"):
                monkeypatch.setattr(ops, route, lambda *a: False)
            monkeypatch.setattr(
                ops, "linear_in_order", lambda x, w, *a, **k: torch.nn.functional.linear(x, w))
        cache, batch = _steps_of(c, lens, cached, decodes, kv)
        logits = model.step(batch, cache)
        assert logits.dtype == torch.float32 and logits.shape == (len(lens) + decodes, 2048)
        rows = [logits]
        for i, pages in enumerate(cache.k_caches + cache.v_caches):
            x = pages
            if cache.fp8:
                scale = (cache.k_scales + cache.v_scales)[i]
                x = pages.view(torch.float8_e4m3fn).float() * scale.unsqueeze(-1)
            rows.append(x.transpose(1, 2).reshape(-1, 2 * D)[batch.slot_mapping].float())
        got.append(rows)
    for one, other in zip(*got):
        # two layers, each of whose ten roundings is 2^-9; a row in e4m3 2^-4
        diff = (one - other).norm() / other.norm()
        assert float(diff) < (0.05 if kv == "fp8" else 0.02), float(diff)


# a wave, 64 to 1024 threads a row, and pieces: the ends of each
@pytest.mark.parametrize("T", [1, 5, 512, 513, 1025])
@pytest.mark.parametrize("H", [8, 504, 512, 520, 1024, 1032, 2056, 4096, 4104, 8192, 8200])
def test_rmsnorm_rows(T, H):
    g = torch.Generator(device=DEV).manual_seed(T + H)
    x, r = ((torch.randn(T, H, generator=g, device=DEV) * 2).bfloat16() for _ in range(2))
    w = torch.randn(H, generator=g, device=DEV).bfloat16()

    def norm(v):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-5) * w.double()

    # half a unit of bf16, fp32 sums of H squares
    near = dict(rtol=2**-8 + 2**-20, atol=1e-6)
    torch.testing.assert_close(ops.rmsnorm(x, w, 1e-5).double(), norm(x.double()), **near)
    total = (x.float() + r.float()).bfloat16()
    y, kept = ops.rmsnorm_residual(x, r, w, 1e-5)
    assert torch.equal(kept, total)
    torch.testing.assert_close(y.double(), norm(total.double()), **near)


# 256 and 512 threads with two pieces each: ends inside the first, the second and
# a later turn
@pytest.mark.parametrize("I", [8, 2040, 4096, 4104, 8200, 14336, 18952])
def test_swiglu_rows(I):
    x = torch.randn(3, 2 * I, generator=torch.Generator(device=DEV).manual_seed(I), device=DEV)
    x = x.bfloat16()
    gate, up = x.double().chunk(2, -1)
    # half a unit of bf16, and an exponential and a quotient in fp32
    torch.testing.assert_close(
        ops.swiglu(x).double(), torch.nn.functional.silu(gate) * up, rtol=2**-8 + 1e-5, atol=1e-30)
