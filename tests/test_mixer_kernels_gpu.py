"""The mechanisms of libslm_mixers one by one against the plain restatement (oracle/vebusun.py): recurrences, their norm and
gate, windowed attention in its three kernels; and the tanh norm, scaled adds and the SiLU GLU of the dense path."""
import numpy as np
import pytest
import torch

from .vebusun_common import lightning, mixer_weights, parallel, random_tensors, window
from oracle import vebusun as ref

pytestmark = pytest.mark.gpu
BOTH = [torch.float32, torch.bfloat16]
DEV = "cuda"


def _close(got, want, dtype, f32=2e-5, b16=4e-2):
    got = got.double().cpu().numpy() if isinstance(got, torch.Tensor) else got
    # (the largest difference over the root mean square: a value five times that, rounded to 16 bits, is off by 0.02 already)
    err = np.abs(got - want).max() / max(np.sqrt((want * want).mean()), 1e-30)
    assert err < (f32 if dtype == torch.float32 else b16), err


def _f64(w):
    return {k: v.double().numpy() for k, v in w.items()}


class _Batch:
    """Steps of one layer over sequences: entries [(sequence, rows)] -> positions and parameters."""

    def __init__(self, n_blocks=40, block_size=16, n_states=5):
        from scalellm_amd.engine import BlockAllocator, StepBuilder
        from scalellm_amd.registry import ModelLimits
        self.allocator = BlockAllocator(n_blocks, block_size, n_states)
        self.builder = StepBuilder(self.allocator, DEV, 2)
        self.limits = lambda dtype: ModelLimits(n_blocks, block_size, dtype, DEV, n_states)

    def run(self, mixer, cache, streams, entries):
        """streams: name -> hidden rows; entries: [(sequence, n)].  -> the mixer's output per entry."""
        step = self.builder.build(entries)
        h = torch.cat([streams[entries[i][0].id][entries[i][0].n_cached:entries[i][0].n_cached + entries[i][1]] for i in step.order])
        out = mixer(h, step.positions, cache, step.params)
        self.builder.commit(entries)
        return [out[step.row0[i]:step.row0[i] + n] for i, (_, n) in enumerate(entries)]


def _total(delta):
    return delta.t.sum(0) if hasattr(delta, "t") and not isinstance(delta, torch.Tensor) else delta.float()


def _hidden(n, width, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(n, width, generator=g).to(torch.bfloat16)
    pad = torch.zeros(n, (width + 63) // 64 * 64)
    pad[:, :width] = h.float()
    return h.double().numpy(), pad.to(device=DEV, dtype=dtype)


def _serve(layer, width, dtype, want_of, eps):
    """Streams of several lengths in uneven portions and single rows, slots used again; every row against want_of(h)."""
    from scalellm_amd.engine import Sequence
    b = _Batch()
    cache = layer.new_cache(b.limits(dtype))
    rng = np.random.default_rng(0)
    streams, want, got, live = {}, {}, {}, []
    for i, n in enumerate((70, 33, 150, 2, 1, 41)):
        h, streams[i] = _hidden(n, width, dtype, 20 + i)
        want[i], got[i] = want_of(h), []
    waiting = [Sequence(i, [0] * streams[i].size(0)) for i in streams]
    while live or waiting:
        while waiting and len(live) < 3:
            live.append(waiting.pop(0))
        entries = [(s, min(len(s.tokens) - s.n_cached, 1 if rng.random() < 0.4 else int(rng.integers(2, 50)))) for s in live]
        for (s, _), o in zip(entries, b.run(lambda *a: _total(layer.forward(*a)), cache, streams, entries)):
            got[s.id].append(o[:, :width])
        for s in [s for s in live if s.n_cached == len(s.tokens)]:
            live.remove(s)
            s.release(b.allocator)
    for i in want:
        _close(torch.cat(got[i]), want[i], dtype, 3e-5, 8e-2)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,taps,width", [(1, 1, 1, 1, 1, 16), (4, 2, 20, 13, 3, 77), (2, 2, 64, 64, 2, 64), (3, 1, 100, 65, 6, 50),
                                                               (2, 1, 192, 130, 4, 64), (2, 2, 256, 256, 4, 64), (70, 35, 32, 16, 4, 96)])
def test_channel_delta(heads, kv_heads, dim, vdim, taps, width, dtype):
    from scalellm_amd.mixer_layers import ChannelDelta, ChannelDeltaArgs
    m = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim, "conv": taps}
    w = mixer_weights("channel_delta", m, width, random_tensors(1))
    layer = ChannelDelta(ChannelDeltaArgs(heads, kv_heads, dim, vdim, taps), width, 1e-5, w, dtype, DEV)
    _serve(layer, width, dtype, lambda h: ref.channel_delta(h, _f64(w), m, 1e-5), 1e-5)


# Channels that forget on both sides of 2^-96 a chunk, where what tokens do to each other is one product of factors, or an exponential a term; a chunk has
# some of either, or of the first only.  Sums of 32 bits whatever the way: the bound is test_channel_delta's.
@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("dim", [20, 128, 200])
@pytest.mark.parametrize("faster", [(6.0, 0.0, 3.5), (3.0, 4.0, 4.4)])
def test_channel_delta_that_forgets_fast(faster, dim, dtype):
    from scalellm_amd.mixer_layers import ChannelDelta, ChannelDeltaArgs
    m = {"heads": 3, "kv_heads": 3, "dim": dim, "vdim": 40, "conv": 4}
    w = mixer_weights("channel_delta", m, 64, random_tensors(5))
    w["A_log"] = w["A_log"] + torch.tensor(faster, dtype=w["A_log"].dtype)
    layer = ChannelDelta(ChannelDeltaArgs(3, 3, dim, 40, 4), 64, 1e-5, w, dtype, DEV)
    _serve(layer, 64, dtype, lambda h: ref.channel_delta(h, _f64(w), m, 1e-5), 1e-5)


class _Alone:
    """One half of a parallel mixer as a layer of its own."""

    def __init__(self, half, width, is_window):
        from scalellm_amd import latent_kernels as lk
        self.half, self.is_window, self.lk, self.width = half, is_window, lk, width

    def new_cache(self, limits):
        return self.half.new_cache(limits) if self.is_window else self.half.new_state(limits)

    def forward(self, h, positions, cache, params):
        proj = self.lk.linear(h, self.half.w_in)
        out = proj.new_full((h.size(0), self.half.out_width + 8), float("nan"))
        self.half.forward(proj, positions, cache, params, out[:, :self.half.out_width])
        return out[:, :self.half.out_width].float() @ self.half.w_o.float().t()


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("dim,vdim,decay", [(1, 1, (0.5,)), (11, 7, (0.3, 0.9, 0.99)), (64, 64, (1.0, 0.999)), (130, 200, (0.97, 0.0)),
                                            (256, 256, (0.9,)), (32, 48, tuple(0.5 + 0.007 * i for i in range(70)))])
def test_lightning_attention(dim, vdim, decay, dtype):
    from scalellm_amd.mixer_layers import LightningArgs, LightningAttention
    _, m = parallel(window(1, 1, 8, 8, 4, 5, 1), lightning(dim, vdim, decay))
    width = 80
    w = {k[6:]: v for k, v in mixer_weights("parallel", m, width, random_tensors(2)).items() if k.startswith("right.")}
    half = LightningAttention(LightningArgs(len(decay), dim, vdim, decay), width, 1e-5, w, dtype, DEV, 0.75)
    _serve(_Alone(half, width, False), width, dtype, lambda h: 0.75 * ref.lightning_attention(h, _f64(w), m["right"], 1e-5), 1e-5)


@np.errstate(over="ignore")
def _lightning_by_hand(proj, H, D, V, decay, weight, eps):
    """The layer behind its projections [q | k | v | g], token by token in 64 bits."""
    x = proj.double().cpu().numpy()
    act = lambda z: z * ref.sigmoid(z)  # noqa: E731
    S, out, qk = np.zeros((H, D, V)), [], H * D
    for r in x:
        q, k, v = act(r[:qk]).reshape(H, D), act(r[qk:2 * qk]).reshape(H, D), act(r[2 * qk:2 * qk + H * V]).reshape(H, V)
        S = np.asarray(decay)[:, None, None] * S + k[:, :, None] * v[:, None, :]
        o = np.einsum("hdv,hd->hv", S, q).reshape(-1)
        out.append(ref.rms_norm(o, weight, eps) * ref.sigmoid(r[2 * qk + H * V:2 * qk + 2 * H * V]))
    return np.array(out)


def _lightning_of(proj, H, D, V, decay, dtype):
    """The same rows as one portion and one by one."""
    from scalellm_amd.engine import Sequence
    from scalellm_amd.mixer_layers import LightningArgs, LightningAttention
    w = {n: torch.zeros(H * d, 64) for n, d in (("q", D), ("k", D), ("v", V), ("g", V))}
    half = LightningAttention(LightningArgs(H, D, V, decay), 64, 1e-5, {**w, "norm": torch.ones(H * V), "o": torch.zeros(64, H * V)}, dtype, DEV)
    got = []
    for n in (proj.size(0), 1):
        b = _Batch()
        state, seq, rows = half.new_state(b.limits(dtype)), Sequence(0, [0] * proj.size(0)), []

        def layer(x, *how):
            out = x.new_empty(x.size(0), half.out_width)
            half.forward(x, *how, out)
            return out
        while seq.n_cached < proj.size(0):
            rows += b.run(layer, state, {0: proj}, [(seq, n)])
        got.append(torch.cat(rows))
    return got


# 16-bit inputs go down to -3e38, and what an activation makes of them is 0 whether a token comes alone or in a portion
@pytest.mark.parametrize("dtype", BOTH)
def test_activations_of_values_far_below_zero(dtype):
    H, D, V, decay = 2, 32, 48, (0.9, 0.6)
    g = torch.Generator().manual_seed(12)
    proj = torch.randn(37, 2 * H * (D + V), generator=g)
    for i, z in enumerate((-3e38, -1e30, -1e28, -1000.0, -90.0, -75.0, -69.5, -60.0)):
        for at in (0, H * D, 2 * H * D):   # of q, k and v
            proj[:, at + 3 * i] = z
            proj[i, at + 30] = z
    proj = proj.to(device=DEV, dtype=dtype)
    want = _lightning_by_hand(proj, H, D, V, decay, 1.0, 1e-5)
    for got in _lightning_of(proj, H, D, V, decay, dtype):
        _close(got, want, dtype, 3e-5, 4e-2)


# Keys are not normed: large ones in a head that forgets almost 2^-96 a chunk, and much more (where a product of exponentials would leave the range).
# (The norm behind squares read-outs, so those stay under 1e19 here: keys of 1e16 make some of 1e17.)
@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("size", [1e12, 1e16])
def test_lightning_attention_of_large_keys(size, dtype):
    H, D, V, decay = 3, 32, 48, (0.0167, 0.9, 1e-6)
    g = torch.Generator().manual_seed(13)
    proj = torch.randn(37, 2 * H * (D + V), generator=g)
    proj[:, H * D:2 * H * D] *= size
    proj = proj.to(device=DEV, dtype=dtype)
    want = _lightning_by_hand(proj, H, D, V, decay, 1.0, 1e-5)
    for got in _lightning_of(proj, H, D, V, decay, dtype):
        _close(got, want, dtype, 3e-5, 4e-2)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("m", [window(1, 1, 2, 1, 2, 1, 0), window(6, 3, 22, 18, 10, 21, 5, 5.0), window(4, 4, 64, 96, 64, 16, 16),
                               window(34, 2, 128, 64, 0, 40, 70, 8.0), window(3, 1, 96, 192, 50, 0, 0, 0.0), window(2, 2, 256, 256, 128, 33, 3),
                               window(2, 1, 200, 128, 200, 64, 1, 3.0), window(2, 1, 300, 260, 40, 30, 4)])
def test_window_attention(m, dtype):
    from scalellm_amd.latent_layers import rotary_table
    from scalellm_amd.mixer_layers import WindowAttention, WindowAttentionArgs
    width = 72
    _, both = parallel(m, lightning(4, 4, (0.5,)))
    w = {k[5:]: v for k, v in mixer_weights("parallel", both, width, random_tensors(3), sharp=1.5).items() if k.startswith("left.")}
    rot = m["rot"]
    args = WindowAttentionArgs(m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["scale"], rot["base"], rot["dims"], m["softcap"],
                               m["mask"]["size"], m["mask"]["keep_first"])
    half = WindowAttention(args, width, 1e-5, w, rotary_table(rot["base"], rot["dims"], 256, device=DEV), dtype, DEV, 1.25)
    _serve(_Alone(half, width, True), width, dtype, lambda h: 1.25 * ref.sink_attention(h, _f64(w), m, 1e-5), 1e-5)


@pytest.mark.parametrize("softcap,sink", [(0.0, False), (6.0, True), (0.0, True)])
@pytest.mark.parametrize("size,keep", [(0, 0), (200, 0), (100, 40), (3, 2)])
@pytest.mark.parametrize("heads,kv_heads,D,V", [(8, 2, 128, 128), (40, 2, 64, 96)])
def test_attention_kernels_agree(heads, kv_heads, D, V, size, keep, softcap, sink):
    """Single rows by the any-size kernel, by MFMA with one and with many splits, and as portions, against the sums written
    out; unequal contexts, blocks in random order, one key per head that stands out just inside or outside the window."""
    from scalellm_amd import mixer_kernels as mk
    from scalellm_amd.layers import InputParameters, Portion
    from scalellm_amd.mixer_layers import WindowPlan
    g = torch.Generator().manual_seed(4)
    B, lens = 16, [1, 17, 700, 64, 333]
    nb = [(n + B - 1) // B for n in lens]
    perm = torch.randperm(sum(nb), generator=g).to(torch.int32) * B
    cu = np.concatenate([[0], np.cumsum(nb)])
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    kc, vc = r(sum(nb) * B, kv_heads, D), r(sum(nb) * B, kv_heads, V)
    q = r(len(lens), heads * D)
    slot = lambda s, j: int(perm[cu[s] + j // B]) + j % B  # noqa: E731
    for s, n in enumerate(lens):      # loud keys around the window's edge and the kept tokens' end
        for j in {n - size, n - size - 1, keep - 1, keep}:
            if 0 <= j < n:
                for a in range(kv_heads):
                    kc[slot(s, j), a] = q[s].view(heads, D)[a * (heads // kv_heads)] * 0.8
    sk = torch.randn(heads, generator=g) + 2 if sink else None
    scale, f = D ** -0.5, 0.5
    want = np.zeros((len(lens), heads, V))
    for s, n in enumerate(lens):
        js = ref.visible(n - 1, {"size": size, "keep_first": keep})
        at = [slot(s, j) for j in js]
        for h in range(heads):
            x = kc[at, h // (heads // kv_heads)].double().numpy() @ q[s].view(heads, D)[h].double().numpy() * scale
            x = softcap * np.tanh(x / softcap) if softcap else x
            p = np.exp(x - x.max())
            extra = np.exp(float(sk[h]) - x.max()) if sink else 0.0
            want[s, h] = f * (p @ vc[at, h // (heads // kv_heads)].double().numpy()) / (p.sum() + extra)
    dev = lambda t: t.to(DEV)  # noqa: E731
    i32 = lambda x: torch.tensor(np.asarray(x), dtype=torch.int32, device=DEV)  # noqa: E731
    q, kc, vc, table, sk = dev(q), dev(kc), dev(vc), dev(perm), None if sk is None else dev(sk)
    how = dict(heads=heads, window=size, keep_first=keep, scale=scale, softcap=softcap, out_scale=f)
    for kw in (dict(generic=True), dict(n_splits=1), dict(n_splits=3), dict(n_splits=7), dict()):
        out = torch.full((len(lens), heads * V), float("nan"), dtype=torch.bfloat16, device=DEV)
        mk.window_attention(q, kc, vc, out, sk, i32(lens) - 1, i32(range(len(lens) + 1)), table, i32(cu), block_size=B, max_kv_len=max(lens),
                            **how, **kw)
        _close(out.view(len(lens), heads, V), want, torch.bfloat16, b16=4e-2)
    ps = [Portion(s, 1, n, perm[cu[s]:cu[s + 1]].numpy()) for s, n in enumerate(lens)]
    prm = InputParameters(*[None] * 5, portions=ps)
    plan = WindowPlan.of(prm, size, keep, B, DEV)
    out = torch.full((len(lens), heads * V), float("nan"), dtype=torch.bfloat16, device=DEV)
    mk.window_prefill(q, kc, vc, out, sk, plan.slots, plan.tiles, **how)
    _close(out.view(len(lens), heads, V), want, torch.bfloat16, b16=4e-2)


@pytest.mark.parametrize("D,V", [(128, 128), (64, 64), (96, 128), (192, 64), (64, 192), (192, 128), (256, 256), (96, 192), (192, 96), (64, 256),
                                 (256, 96), (256, 192)])   # (the wide ones but 256 / 256: tiles of 32 keys; of 96 columns the last load is of two waves)
@pytest.mark.parametrize("size,keep,softcap,sink", [(0, 0, 0.0, False), (150, 70, 6.0, True), (40, 0, 6.0, False), (0, 0, 50.0, True)])
def test_portions_with_and_without_shared_tiles(D, V, size, keep, softcap, sink):
    """Few workgroups (two groups of waves share a portion's tiles) and many (one group), at the edges of the tiles of 64 keys
    and 128 rows, the fewest shared tiles, odd and even numbers of them."""
    from scalellm_amd import mixer_kernels as mk
    from scalellm_amd.layers import InputParameters, Portion
    from scalellm_amd.mixer_layers import WindowPlan
    g = torch.Generator().manual_seed(6)
    B, heads, kv_heads = 16, 32, 8
    spans = [(1, 1), (64, 64), (65, 65), (129, 129), (5, 260), (200, 320), (31, 321), (130, 449), (400, 600), (2, 500), (3, 1000)]   # rows, context
    nb = [(k + B - 1) // B for _, k in spans]
    perm = torch.randperm(sum(nb), generator=g).to(torch.int32) * B
    cu = np.concatenate([[0], np.cumsum(nb)])
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
    kc, vc, q = r(sum(nb) * B, kv_heads, D), r(sum(nb) * B, kv_heads, V), r(sum(n for n, _ in spans), heads * D)
    sk = (torch.randn(heads, generator=g) + 2).to(DEV) if sink else None
    how = dict(heads=heads, window=size, keep_first=keep, scale=2 * D ** -0.5, softcap=softcap, out_scale=0.5)
    portions, want, row = [], [], 0
    for i, (n, k) in enumerate(spans):
        portions.append(Portion(row, n, k, perm[cu[i]:cu[i + 1]].numpy()))
        j = torch.arange(k)
        at = (perm[cu[i] + j // B].long() + j % B).to(DEV)
        pos, j = torch.arange(k - n, k, device=DEV)[:, None], j.to(DEV)[None]
        seen = (j <= pos) & ((pos - j < size) | (j < keep) if size else True)
        for h in range(heads):
            x = q[row:row + n, h * D:(h + 1) * D].double() @ kc[at, h // 4].double().t() * how["scale"]
            x = (softcap * torch.tanh(x / softcap) if softcap else x).masked_fill(~seen, -float("inf"))
            if sink:
                x = torch.cat([x, sk[h].double().expand(n, 1)], 1)
            want.append(0.5 * (torch.softmax(x, 1)[:, :k] @ vc[at, h // 4].double()))
        row += n
    got = {}
    for many in (False, True):
        out = torch.full((row, heads * V), float("nan"), dtype=torch.bfloat16, device=DEV)
        for ps in ([portions] if many else [[p] for p in portions]):   # 17 tiles of 32 heads, and up to 4
            plan = WindowPlan.of(InputParameters(*[None] * 5, portions=ps), size, keep, B, DEV)
            assert len(plan.tiles) * heads > 512 if many else len(plan.tiles) * heads <= 256   # (between them the contexts decide)
            mk.window_prefill(q, kc, vc, out, sk, plan.slots, plan.tiles, **how)
        got[many] = out.double()
    for i, (n, _) in enumerate(spans):
        for h in range(heads):
            w, p0 = want[i * heads + h], portions[i].row0
            for out in got.values():   # 16-bit weights and results: 2^-9 of each, relative to the row
                assert ((out[p0:p0 + n, h * V:(h + 1) * V] - w).norm(dim=1) <= 2.0 ** -7 * w.norm(dim=1) + 2.0 ** -8).all()


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("per_head", [True, False])
@pytest.mark.parametrize("heads,vdim", [(1, 1), (3, 13), (16, 128), (5, 200)])
def test_gated_norm(heads, vdim, per_head, dtype):
    from scalellm_amd import mixer_kernels as mk
    g = torch.Generator().manual_seed(5)
    rows, v_pad, n = 9, (vdim + 15) // 16 * 16, heads * vdim
    o = torch.randn(rows, heads, v_pad, generator=g) * 3
    gate = torch.randn(rows, n + 8, generator=g).to(dtype)
    w = torch.randn(vdim if per_head else n, generator=g)
    out = torch.full((rows, n + 24), float("nan"), dtype=dtype, device=DEV)
    mk.gated_norm(o.to(DEV), vdim, gate.to(DEV), w.to(DEV), out, eps=1e-3, per_head=per_head, scale=0.3)
    x = o[:, :, :vdim].double().numpy()
    x = x if per_head else x.reshape(rows, n)
    want = 0.3 * ref.rms_norm(x, w.double().numpy(), 1e-3).reshape(rows, n) * ref.sigmoid(gate[:, :n].double().numpy())
    _close(out[:, :n], want, dtype)
    assert float(out[:, n:].abs().max()) == 0.0


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("width,rows", [(33, 5), (256, 3), (2048, 40)])
def test_tanh_norm_and_scaled_adds(width, rows, dtype):
    from scalellm_amd import latent_kernels as lk
    g = torch.Generator().manual_seed(6)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    w, b, alpha, mult, ld = r(width), r(width), 0.7, 0.3, (width + 63) // 64 * 64
    norm = lk.TanhNorm(alpha, w.to(DEV), b.to(DEV))
    plain = lambda x: ref.dynamic_tanh(x, alpha, w.double().numpy(), b.double().numpy())  # noqa: E731

    def check(x, resid, out):
        _close(resid, x, torch.float32, 1e-6)
        _close(out[:, :width], plain(x), dtype, 1e-5, 3e-2)
        assert ld == width or float(out[:, width:].abs().max()) == 0.0
    table, tokens = r(20, width).to(dtype), torch.arange(rows, dtype=torch.int32) % 20
    resid = torch.empty(rows, width, device=DEV)
    out = torch.empty(rows, ld, dtype=dtype, device=DEV)
    lk.residual_norm(resid, out, norm, 0.0, embed=(tokens.to(DEV), table.to(DEV), None, None), mult=4.5)
    x = table.double().numpy()[tokens.numpy()] * 4.5
    check(x, resid, out)
    delta = r(rows, ld).to(dtype)
    lk.residual_norm(resid, out, norm, 0.0, delta=delta.to(DEV), mult=mult)
    x = x + mult * delta[:, :width].double().numpy()
    check(x, resid, out)
    slabs = r(11, rows, ld)
    lk.residual_norm(resid, out, norm, 0.0, delta=lk.Slabs(slabs.to(DEV)), mult=mult)
    x = x + mult * slabs.double().sum(0)[:, :width].numpy()
    check(x, resid, out)
    pick = torch.tensor([rows - 1, 0], dtype=torch.int32, device=DEV)
    out = torch.empty(2, ld, dtype=dtype, device=DEV)
    lk.residual_norm(resid, out, norm, 0.0, row_index=pick)
    _close(out[:, :width], plain(x[[rows - 1, 0]]), dtype, 1e-5, 3e-2)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("rows", [1, 20, 70])
def test_silu_glu(rows, dtype):
    from scalellm_amd.latent_layers import ClampedGLU
    rnd, W, ff = random_tensors(7), 60, 90
    w = {"gate": rnd(ff, W, std=0.5), "up": rnd(ff, W, std=0.5), "down": rnd(W, ff, std=0.1)}
    h, x = _hidden(rows, W, dtype, 8)
    layer = ClampedGLU(W, ff, float("inf"), w, dtype, DEV, 1.0, 0.0)
    _close(_total(layer.forward(x))[:, :W], ref.feed_forward(h, _f64(w)), dtype, 1e-5, 3e-2)


# few workgroups, enough and many: 1, 2 and 4 kv heads in a workgroup, 4, 2 and 1 of its waves on each; odd counts of
# kv heads, more than 16 query heads on one, ranges of less than a tile, of splits that get no tile, windows with kept tokens
@pytest.mark.parametrize("rows,heads,kv_heads,dim,vdim,longest,window,keep", [
    (3, 6, 3, 64, 128, 900, 0, 0), (40, 8, 2, 128, 128, 300, 100, 7), (130, 16, 4, 96, 64, 200, 0, 0), (9, 160, 8, 128, 128, 700, 0, 0),
    (130, 20, 5, 64, 64, 65, 33, 40), (64, 8, 8, 128, 128, 1500, 1000, 16), (1, 8, 8, 128, 128, 4000, 0, 0),
    (260, 8, 8, 64, 64, 200, 0, 0),    # (four heads, one split)
    (130, 16, 8, 128, 128, 130, 0, 0), (40, 8, 2, 64, 64, 1700, 0, 0), (70, 64, 2, 64, 128, 1100, 0, 0)])   # (two heads: one split, several, blocks of heads)
def test_window_attention_of_single_rows(rows, heads, kv_heads, dim, vdim, longest, window, keep):
    from scalellm_amd import mixer_kernels as mk
    from scalellm_amd.decode import make_batch_inputs
    g = torch.Generator().manual_seed(rows)
    lens = [1, longest] + torch.randint(1, longest + 1, (rows,), generator=g).tolist()
    lens = lens[:rows] if rows > 1 else [longest]
    _, positions, params, n_blocks = make_batch_inputs([1] * rows, lens, 16, DEV, seed=2)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
    q, k, v, sink = rnd(rows, heads * dim), rnd(n_blocks * 16, kv_heads, dim), rnd(n_blocks * 16, kv_heads, vdim), rnd(heads).float()
    out = torch.zeros(rows, heads * vdim, dtype=torch.bfloat16, device=DEV)
    mk.window_attention(q, k, v, out, sink, positions, params.q_cu_seq_lens, params.block_tables, params.cu_block_lens, block_size=16,
                        max_kv_len=longest, heads=heads, window=window, keep_first=keep, scale=dim ** -0.5, softcap=20.0, out_scale=0.7)
    table, starts, group = params.block_tables.long(), params.cu_block_lens.tolist(), heads // kv_heads
    want = torch.empty(rows, heads, vdim, dtype=torch.float64, device=DEV)
    for r, n in enumerate(lens):
        pos = torch.arange(n, device=DEV)
        if window:
            pos = pos[(n - 1 - pos < window) | (pos < keep)]
        slots = table[starts[r] + pos // 16] + pos % 16
        ks, vs = k[slots].double(), v[slots].double()
        for h in range(heads):
            s = ks[:, h // group] @ q[r, h * dim:(h + 1) * dim].double() * dim ** -0.5
            s = 20.0 * torch.tanh(s / 20.0)
            e = torch.exp(s)
            want[r, h] = 0.7 * (e @ vs[:, h // group]) / (e.sum() + torch.exp(sink[h].double()))
    got = out.view(rows, heads, vdim).double()
    # bf16 soft-max weights and results: 2^-9 each of a value, relative to the row
    assert ((got - want).norm(dim=-1) / want.norm(dim=-1)).max() < 1e-2


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("per_head", [True, False])
@pytest.mark.parametrize("rows,heads,vdim,shift", [(1, 1, 64, 0), (33, 3, 64, 0), (70, 7, 64, 0), (70, 2, 256, 0), (17, 5, 128, 0), (9, 32, 256, 0), (9, 33, 256, 0),
                                                   (5, 4, 128, 4)])
def test_gated_norm_of_eights(rows, heads, vdim, shift, per_head, dtype):
    """Workgroups that end within a row, rows of 8192 (the most registers hold) and above, a gate off its 16 bytes in bf16."""
    from scalellm_amd import mixer_kernels as mk
    g = torch.Generator().manual_seed(7)
    n = heads * vdim
    o = torch.randn(rows, heads, vdim, generator=g) * 3
    gate = torch.randn(rows, n + 8 + shift, generator=g).to(dtype).to(DEV)[:, shift:]
    w = torch.randn(vdim if per_head else n, generator=g)
    out = torch.full((rows, n + 40), float("nan"), dtype=dtype, device=DEV)
    mk.gated_norm(o.to(DEV), vdim, gate, w.to(DEV), out, eps=1e-3, per_head=per_head, scale=0.3)
    x = o.double().numpy() if per_head else o.double().numpy().reshape(rows, n)
    want = 0.3 * ref.rms_norm(x, w.double().numpy(), 1e-3).reshape(rows, n) * ref.sigmoid(gate[:, :n].double().cpu().numpy())
    # (one rounding to bf16, whose neighbours above 1 are 2^-7 apart: half of that, 2^-8 of the value at most)
    got = out[:, :n].double().cpu().numpy()
    np.testing.assert_allclose(got, want, rtol=1e-5 if dtype == torch.float32 else 2 ** -8 + 1e-5, atol=1e-6)
    assert float(out[:, n:].abs().max()) == 0.0


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("heads,kv,dim,d_pad,rot,v_pad,shift", [(16, 8, 128, 128, 128, 128, 0), (3, 1, 64, 64, 32, 128, 0),
                                                                (2, 2, 256, 256, 0, 64, 0), (6, 3, 112, 128, 48, 112, 0),
                                                                (4, 2, 128, 128, 24, 128, 0), (4, 2, 64, 64, 64, 64, 4)])
def test_window_append(heads, kv, dim, d_pad, rot, v_pad, shift, dtype):
    """Queries in place and keys and values in their slots: every head width that columns in eights have, a rotation that ends or
    whose halves end within a head, heads narrower than their columns, halves that are no eights, rows off their 16 bytes."""
    from scalellm_amd import mixer_kernels as mk
    g = torch.Generator().manual_seed(8)
    rows, eps, off_k = 21, 1e-3, heads * d_pad
    off_v = off_k + kv * d_pad
    proj = torch.randn(rows, off_v + kv * v_pad + 8 + shift, generator=g).to(dtype)[:, shift:]
    qw, kw, angle = torch.randn(dim, generator=g), torch.randn(dim, generator=g), torch.randn(50, rot // 2, generator=g)
    cs = torch.cat([angle.cos(), angle.sin()], dim=1).contiguous()
    pos, slots = torch.randperm(50, generator=g)[:rows].int(), torch.randperm(40, generator=g)[:rows].int()
    keys = torch.full((40, kv, d_pad), 5.0, dtype=dtype, device=DEV)
    values = torch.full((40, kv, v_pad), 5.0, dtype=dtype, device=DEV)
    x = proj.to(DEV) if not shift else torch.nn.functional.pad(proj, (shift, 0)).to(DEV)[:, shift:]
    mk.window_append(x, keys, values, qw.to(DEV), kw.to(DEV), cs.to(DEV), pos.to(DEV), slots.to(DEV), heads=heads, dim=dim, off_q=0,
                     off_k=off_k, off_v=off_v, eps=eps)
    src, c, s = proj.double().numpy(), np.cos(angle.double().numpy())[pos][:, None], np.sin(angle.double().numpy())[pos][:, None]

    def check(got, v, w, n):
        y = ref.rms_norm(v.reshape(rows, n, d_pad)[:, :, :dim], w.double().numpy(), eps)
        lo, hi = y[:, :, :rot // 2].copy(), y[:, :, rot // 2:rot].copy()
        size = np.abs(y).copy()
        size[:, :, :rot // 2] = size[:, :, rot // 2:rot] = np.hypot(lo, hi)
        y[:, :, :rot // 2], y[:, :, rot // 2:rot] = lo * c - hi * s, lo * s + hi * c
        got = got.double().cpu().numpy().reshape(rows, n, d_pad)
        # (one rounding to bf16, at most 2^-8 of the value; the rotation in 32 bits is off by some 1e-7 of the pair it turns)
        assert (np.abs(got[:, :, :dim] - y) <= (0 if dtype == torch.float32 else 2 ** -8) * np.abs(y) + 2e-6 * size).all()
        assert not got[:, :, dim:].any()
    check(x[:, :off_k], src[:, :off_k], qw, heads)
    check(keys[slots.long()], src[:, off_k:off_v], kw, kv)
    assert torch.equal(values[slots.long()].cpu(), proj[:, off_v:off_v + kv * v_pad].reshape(rows, kv, v_pad))
    assert torch.equal(x[:, off_k:].cpu(), proj[:, off_k:])
    rest = [i for i in range(40) if i not in slots.tolist()]
    assert (keys[rest] == 5.0).all() and (values[rest] == 5.0).all()


@pytest.mark.parametrize("heads,kv,dim,rot,rows", [(3, 1, 64, 32, 999), (3, 1, 64, 32, 1001), (4, 4, 48, 16, 450), (16, 8, 64, 64, 700)])
def test_window_append_of_many_narrow_heads(heads, kv, dim, rot, rows):
    """Heads of 64 go eight columns a lane from some thousands of vectors on: the same as in smaller calls, to a rounding to bf16."""
    from scalellm_amd import mixer_kernels as mk
    g = torch.Generator(device=DEV).manual_seed(9)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=DEV)  # noqa: E731
    off_k = heads * 64
    off_v = off_k + kv * 64
    proj = rnd(rows, off_v + kv * 64).to(torch.bfloat16)
    for t, n in ((proj[:, :off_k], heads), (proj[:, off_k:off_v], kv)):
        t.view(rows, n, 64)[..., dim:] = 0.0
    qw, kw, cs = rnd(dim), rnd(dim), rnd(50, rot)
    pos, slots = torch.randint(0, 50, (rows,), generator=g, device=DEV).int(), torch.randperm(rows, generator=g, device=DEV).int()
    got = []
    for step in (rows, 100):
        x, keys, values = proj.clone(), *(torch.full((rows, kv, 64), 5.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        for r in range(0, rows, step):
            mk.window_append(x[r:r + step], keys, values, qw, kw, cs, pos[r:r + step], slots[r:r + step], heads=heads, dim=dim, off_q=0,
                             off_k=off_k, off_v=off_v, eps=1e-3)
        got.append((x[:, :off_k].float(), keys.float(), values.float()))
    assert torch.equal(got[0][2], got[1][2])
    for a, b in zip(got[0][:2], got[1][:2]):   # (32-bit sums in another order: neighbouring bf16 values at most, 2^-7 of a value apart)
        assert ((a - b).abs() <= 2 ** -7 * torch.maximum(a.abs(), b.abs()) + 1e-5).all() and (a - b).norm() <= 1e-3 * b.norm()
