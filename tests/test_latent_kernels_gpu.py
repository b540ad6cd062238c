"""The mechanisms of the dense / latent-attention library one by one against plain double-precision arithmetic."""
import numpy as np
import pytest
import torch

from oracle import dagupel as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = [torch.float32, torch.bfloat16]


def _lk():
    from scalellm_amd import latent_kernels
    return latent_kernels


def _rnd(seed, *shape, dtype=torch.float32, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(dtype).to(DEV)


def _f64(t):
    return t.detach().double().cpu().numpy()


def _close(got, want, dtype, f32=3e-6, b16=1e-2):
    got, want = _f64(got), np.asarray(want, dtype=np.float64)
    assert got.shape == want.shape and np.isfinite(got).all()
    err = np.abs(got - want).max() / max(np.abs(want).max(), 1e-30)
    assert err < (f32 if dtype == torch.float32 else b16), err


# ---- residual stream and norm ------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,width", [(1, 64), (5, 77), (3, 4096), (130, 100), (2, 7168), (255, 2048), (256, 2048), (2, 2044), (3, 16384), (257, 2500)])
def test_residual_norm_modes(rows, width, dtype):
    lk, eps = _lk(), 1e-5
    pad = (width + 63) // 64 * 64
    w = _rnd(1, width)
    table, pos = _rnd(2, 32, pad, dtype=dtype), _rnd(3, 50, width, dtype=dtype)
    tokens = torch.randint(0, 32, (rows,), dtype=torch.int32, device=DEV)
    positions = torch.randint(0, 50, (rows,), dtype=torch.int32, device=DEV)
    resid = torch.full((rows, width), float("nan"), device=DEV)
    out = torch.full((rows, pad), 7.0, dtype=dtype, device=DEV)

    def check(x):
        np.testing.assert_allclose(_f64(resid), x, rtol=1e-6, atol=1e-6 * np.abs(x).max())
        _close(out[:, :width], ref.rms_norm(x, _f64(w), eps), dtype)
        assert not out[:, width:].any()
    x = _f64(table)[_f64(tokens).astype(int), :width]
    lk.residual_norm(resid, out, w, eps, embed=(tokens, table, None, None))
    check(x)
    x = x + _f64(pos)[_f64(positions).astype(int)]
    lk.residual_norm(resid, out, w, eps, embed=(tokens, table, positions, pos))
    check(x)
    delta = _rnd(4, rows, pad, dtype=dtype)
    lk.residual_norm(resid, out, w, eps, delta=delta)
    x = x + _f64(delta)[:, :width]
    check(x)
    slabs = _rnd(5, 3, rows, pad)
    lk.residual_norm(resid, out, w, eps, delta=lk.Slabs(slabs))
    x = x + _f64(slabs).sum(0)[:, :width]
    check(x)
    lk.residual_norm(resid, out, None, eps, delta=delta)      # the sum only
    x = x + _f64(delta)[:, :width]
    np.testing.assert_allclose(_f64(resid), x, rtol=1e-6, atol=2e-6 * np.abs(x).max())
    pick = torch.tensor([rows - 1, 0, rows // 2], dtype=torch.int32, device=DEV)
    out = torch.full((3, pad), 7.0, dtype=dtype, device=DEV)
    lk.residual_norm(resid, out, w, eps, row_index=pick)
    _close(out[:, :width], ref.rms_norm(x[[rows - 1, 0, rows // 2]], _f64(w), eps), dtype)


def test_residual_norm_of_rows_before_the_named_ones():
    lk = _lk()
    resid, w = _rnd(1, 9, 256), _rnd(2, 256)
    picked, shifted = torch.empty(3, 256, device=DEV), torch.empty(3, 256, device=DEV)
    ends = torch.tensor([0, 3, 4, 9], dtype=torch.int32, device=DEV)
    lk.residual_norm(resid, picked, w, 1e-5, row_index=ends[1:] - 1)
    lk.residual_norm(resid, shifted, w, 1e-5, row_index=ends[1:], row_shift=-1)
    assert torch.equal(picked, shifted)


def test_eps_is_inside_the_root():
    lk = _lk()
    x = torch.full((1, 64), 1e-3, device=DEV)
    out = torch.empty(1, 64, device=DEV)
    lk.residual_norm(x, out, torch.ones(64, device=DEV), 1e-2)
    np.testing.assert_allclose(_f64(out), 1e-3 / np.sqrt(1e-6 + 1e-2), rtol=1e-6)


# ---- products ----------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (3, 48, 320), (16, 80, 1024), (17, 112, 192), (33, 96, 2048), (64, 272, 128),
                                   (65, 64, 64), (200, 144, 256), (1, 4096, 4096),
                                   (30, 16416, 128), (20, 4096, 8192), (50, 16416, 64)])
def test_linear_epilogues(M, N, K, dtype):
    lk = _lk()
    x, w = _rnd(1, M, K, dtype=dtype), _rnd(2, N, K, dtype=dtype, std=K ** -0.5)
    want = _f64(x) @ _f64(w).T
    _close(lk.linear(x, w), want, dtype, f32=1e-5)
    _close(lk.linear_f32(x, w, 0.25), 0.25 * want, torch.float32, f32=1e-5)
    s = lk.linear_slabs(x, w)
    _close(s.t.sum(0), want, torch.float32, f32=1e-5)
    if N % 32 == 0:
        out = torch.empty(M, N // 2, dtype=dtype, device=DEV)
        lk.linear_glu(x, w, out, 0.6)
        _close(out, ref.clamped_glu(want[:, :N // 2], want[:, N // 2:], 0.6), dtype, f32=1e-5, b16=2e-2)


@pytest.mark.parametrize("N,K", [(0, 128), (48, 0)])
def test_products_of_many_rows_of_nothing(N, K):
    lk = _lk()
    for M in (100, 200):
        y = lk.linear(torch.ones(M, K, dtype=torch.bfloat16, device=DEV), torch.ones(N, K, dtype=torch.bfloat16, device=DEV))
        assert y.shape == (M, N) and not y.any()


# row counts at the edges of every tile, columns that fill no panel of 64 and those that decide between tile widths, step
# counts below and at a ring and a split.  fp32 sums of exact products of bf16: 1e-5 of the largest as above.
@pytest.mark.parametrize("M", [1, 2, 16, 17, 32, 33, 64, 65, 127, 128, 140])
@pytest.mark.parametrize("N,K", [(16, 64), (80, 192), (64, 576), (144, 1088), (192, 2112), (2048, 2048), (7168, 320), (16384, 128),
                                 (16896, 64)])
def test_streamed_products(M, N, K):
    _streamed_products(M, N, K)


# Every tile shape of the dispatch with turns of its steady loop (several rings of steps a wave, or a split of it), in every epilogue that
# it has, and step counts that leave waves, groups of waves and rings unequal tails.
@pytest.mark.parametrize("M", [1, 16, 32, 63, 64, 100, 128, 140])
@pytest.mark.parametrize("N,K", [(28672, 704), (16896, 1088), (16384, 2240), (7168, 1344), (6784, 2112), (1024, 16448), (64, 32832)])
def test_streamed_products_of_many_steps(M, N, K):
    _streamed_products(M, N, K)


# The edges of the 96-row tiles, with columns that make them narrow and wide, and step counts below, at and past their ring.
@pytest.mark.parametrize("M", [80, 96, 97])
@pytest.mark.parametrize("N,K", [(80, 192), (2048, 320), (16896, 256), (28672, 704), (1024, 8256)])
def test_streamed_products_of_96_row_tiles(M, N, K):
    _streamed_products(M, N, K)


def _streamed_products(M, N, K):
    lk = _lk()
    x = _rnd(1, M, K + 8, dtype=torch.bfloat16)[:, :K]
    w = _rnd(2, N, K, dtype=torch.bfloat16, std=K ** -0.5)
    want = _f64(x) @ _f64(w).T
    layout = lk.stream_layout(w)
    _close(lk.linear_f32(x, w, 0.25, layout), 0.25 * want, torch.float32, f32=1e-5)
    _close(lk.linear(x, w, layout=layout), want, torch.bfloat16)
    if 64 < M <= 128:   # (linear() leaves products of so many rows that are only stored to the vendor's: the streamed form by its own entry)
        wide = torch.full((M, N + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
        a = lk._stream_args(x, w, layout, M, N, K, 128)
        a.ldy, a.y, a.epilogue = N + 8, wide.data_ptr(), lk._lib.LIN_STORE
        lk._run_stream(a)
        _close(wide[:, :N], want, torch.bfloat16)
        assert wide[:, N:].isnan().all()
    s = lk.linear_slabs(x, w, layout)
    _close(s.t.sum(0), want, torch.float32, f32=1e-5)
    if N % 64 == 0:
        out = torch.zeros(M, N // 2, dtype=torch.bfloat16, device=DEV)
        lk.linear_glu(x, w, out, 0.6, layout=lk.stream_layout(w, glu=True))
        _close(out, ref.clamped_glu(want[:, :N // 2], want[:, N // 2:], 0.6), torch.bfloat16, b16=2e-2)


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("N,K,n", [(16, 64, 3), (80, 704, 2), (3664, 1984, 3), (6752, 2112, 2), (9216, 1088, 3), (1040, 4160, 16), (16384, 192, 1)])
def test_products_cut_in_k_and_joined(M, N, K, n):
    """Splits without a step, last panels that are not whole, tiles of 32, 64 and 128 columns; the counters are zero again after every launch."""
    lk = _lk()
    from scalellm_amd import _lib
    x, w = _rnd(1, M, K + 8, dtype=torch.bfloat16)[:, :K], _rnd(2, N, K, dtype=torch.bfloat16)
    resid, h, table = torch.empty(1, 64, device="cuda"), torch.empty(1, 64, device="cuda"), torch.ones(1, 64, device="cuda")
    tickets = torch.full((_lib.STREAM_TICKETS,), 7, dtype=torch.int32, device="cuda")
    lk.residual_norm(resid, h, torch.ones(64, device="cuda"), 1e-5, embed=(torch.zeros(1, dtype=torch.int32, device="cuda"), table, None, None), clear=tickets)
    want, outs = _f64(x) @ _f64(w).T, []
    layout = lk.stream_layout(w)
    for _ in range(3):
        out = torch.full((M, N + 4), 9.0, dtype=torch.bfloat16, device="cuda")
        a = lk._stream_args(x, w, layout, M, N, K, 128)
        a.ldy, a.y, a.epilogue = out.stride(0), out.data_ptr(), _lib.LIN_STORE
        assert lk._joined(a, n, tickets, x.device)
        assert int(tickets.abs().max()) == 0
        assert bool((out[:, N:] == 9.0).all())
        outs.append(out[:, :N])
    # one rounding to bf16 (2^-9) of sums whose 32-bit error is far below it
    assert (np.abs(_f64(outs[0]) - want) - np.abs(want) * 2.0 ** -8).max() < 2e-5 * K ** 0.5
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    got = lk.linear(x, w, layout=layout, tickets=lk.StepTickets(tickets))   # (as many as pay, or none)
    assert (np.abs(_f64(got) - want) - np.abs(want) * 2.0 ** -8).max() < 2e-5 * K ** 0.5 and int(tickets.abs().max()) == 0


def test_joined_products_in_a_graph():
    lk = _lk()
    M, N, K = 100, 3664, 2048
    x, w = _rnd(1, M, K, dtype=torch.bfloat16), _rnd(2, N, K, dtype=torch.bfloat16)
    layout, tickets = lk.stream_layout(w), lk.StepTickets(torch.zeros(512, dtype=torch.int32, device="cuda"))
    assert lk.join_count(N, K, M) > 1
    lk.linear(x, w, layout=layout, tickets=tickets)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        first = lk.linear(x, w, layout=layout, tickets=tickets)
        again = lk.linear(first[:, :K], w, layout=layout, tickets=tickets)
    for i in range(4):
        x.copy_(_rnd(3 + i, M, K, dtype=torch.bfloat16))
        graph.replay()
        torch.cuda.synchronize()
        a = lk.linear(x, w, layout=layout, tickets=tickets)
        b = lk.linear(a[:, :K], w, layout=layout, tickets=tickets)
        assert torch.equal(first, a) and torch.equal(again, b)


# Products of many rows, in every tile: rows and columns that fill no tile, one step of 64 k and fewer than there are stages, more tiles than
# CUs with the rest cut in K (also by a count that leaves the last slice short), rows with a stride.  fp32 sums of exact products, one rounding;
# the slices' sums come in a fixed order, so a second run gives the same bits.
@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("M,N,K,slices", [(1, 16, 64, 1), (129, 272, 128, 2), (300, 544, 704, 3), (257, 96, 1088, 5), (160, 1312, 192, 1), (2300, 4128, 320, 2)])
def test_tiled_products(M, N, K, slices, tile):
    lk = _lk()
    x = _rnd(1, M, K + 8, dtype=torch.bfloat16)[:, :K]
    w = _rnd(2, N, K, dtype=torch.bfloat16, std=K ** -0.5)
    want = _f64(x) @ _f64(w).T
    wide = torch.full((M, N + 16), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = wide[:, 8:8 + N]
    assert lk._gemm(x, w, out, tile=tile, slices=slices)
    _close(out, want, torch.bfloat16)
    assert wide[:, :8].isnan().all() and wide[:, 8 + N:].isnan().all()
    again = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
    assert lk._gemm(x, w, again, tile=tile, slices=slices) and torch.equal(again, out)
    if tile != 4 and N % 32 == 0:   # (that tile has no GLU)
        glu = torch.full((M, N // 2 + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert lk._gemm(x, w, glu[:, :N // 2], (0.6, lk.GLU_ALPHA, lk.GLU_SHIFT), tile, slices)
        _close(glu[:, :N // 2], ref.clamped_glu(want[:, :N // 2], want[:, N // 2:], 0.6), torch.bfloat16, b16=2e-2)
        assert glu[:, N // 2:].isnan().all()


# The same in half precision: every tile, rows and columns that fill none, tiles that are cut, and more of them than CUs.
@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("M,N,K,slices", [(1, 32, 64, 1), (300, 544, 704, 3), (2300, 7456, 192, 1)])
def test_tiled_products_in_half_precision(M, N, K, slices, tile):
    lk = _lk()
    x = _rnd(1, M, K + 8, dtype=torch.float16)[:, :K]
    w = _rnd(2, N, K, dtype=torch.float16, std=K ** -0.5)
    want = x.double() @ w.double().t()
    wide = torch.full((M, N + 16), float("nan"), dtype=torch.float16, device=DEV)
    assert lk.gemm(x, w, wide[:, 8:8 + N], None, tile, slices)
    assert (wide[:, 8:8 + N].double() - want).abs().max() <= 2.0 ** -11 * 1.02 * want.abs().max()
    assert wide[:, :8].isnan().all() and wide[:, 8 + N:].isnan().all()
    if tile != 4:   # (that one has no GLU)
        glu = torch.full((M, N // 2 + 8), float("nan"), dtype=torch.float16, device=DEV)
        assert lk.gemm(x, w, glu[:, :N // 2], (0.6, lk.GLU_ALPHA, lk.GLU_SHIFT), tile, slices)
        out = torch.from_numpy(ref.clamped_glu(want[:, :N // 2].cpu().numpy(), want[:, N // 2:].cpu().numpy(), 0.6)).to(DEV)
        assert (glu[:, :N // 2].double() - out).abs().max() <= 2.0 ** -11 * 1.05 * out.abs().max() and glu[:, N // 2:].isnan().all()


# More tiles than CUs, so that a workgroup goes from one to the next: steps at, one and two past the stages that are loaded ahead, two rounds and
# three, a last round that is cut, also so that its last slice is at the stages (then a workgroup has one item, as with K 192 and three of them).
@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("M,N,K,slices", [(2300, 7456, 192, 1), (2300, 7456, 256, 1), (2300, 7456, 320, 1), (1100, 16416, 704, 2), (2300, 8224, 576, 3)])
def test_tiled_products_of_several_rounds(M, N, K, slices, tile):
    test_tiled_products(M, N, K, slices, tile)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,slices,glu", [(257, 96, 1088, 5, False), (300, 544, 704, 3, True), (1100, 16416, 704, 2, False), (207, 4096, 2048, 0, False)])
def test_tiled_products_with_counters_of_the_callers(M, N, K, slices, glu, dtype):
    """The same bits as with counters of the launch's own; eagerly and in a graph."""
    lk = _lk()
    x, w = _rnd(1, M, K, dtype=dtype), _rnd(2, N, K, dtype=dtype, std=K ** -0.5)
    how = dict(glu=(7.0, 1.0, 0.0) if glu else None, slices=slices)
    want, got = (torch.zeros(M, N // 2 if glu else N, dtype=dtype, device="cuda") for _ in range(2))
    words = torch.zeros(512 + 3 * 256, dtype=torch.int32, device="cuda")
    tickets = lk.StepTickets(words)
    assert lk._gemm(x, w, want, **how)
    for _ in range(4):   # (the last one finds none left)
        got.zero_()
        assert lk._gemm(x, w, got, tickets=tickets, **how) and torch.equal(want, got)
    assert int(words[:512].abs().max()) == 0 and bool((words.view(-1, 256)[2:] == words[512:768]).all())
    assert int(words[512:768].max()) > 0   # (it was cut, and counted there)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        words.zero_()
        tickets = lk.StepTickets(words)
        for _ in range(2):
            lk._gemm(x, w, got, tickets=tickets, **how)
    for i in range(3):
        x.copy_(_rnd(3 + i, M, K, dtype=dtype))
        graph.replay()
        lk._gemm(x, w, want, **how)
        assert torch.equal(want, got)


@pytest.mark.parametrize("M", [129, 700])
def test_products_of_prompts_by_the_planned_tile(M):
    lk, N, K = _lk(), 2080, 1024
    x, w = _rnd(1, M, 2 * K, dtype=torch.bfloat16)[:, K:], _rnd(2, N, K, dtype=torch.bfloat16, std=K ** -0.5)
    want, out = _f64(x) @ _f64(w).T, torch.zeros(M, N // 2, dtype=torch.bfloat16, device=DEV)
    _close(lk.linear(x, w), want, torch.bfloat16)
    lk.linear_glu(x, w, out, 0.6)
    _close(out, ref.clamped_glu(want[:, :N // 2], want[:, N // 2:], 0.6), torch.bfloat16, b16=2e-2)
    # without scratch nothing is cut; results are the same up to the order of sums
    from scalellm_amd import _lib
    a = lk._linear_args(x, w, M, N, K)
    y = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
    a.ldx, a.ldw, a.ldy, a.y, a.epilogue = x.stride(0), K, N, lk._p(y), _lib.LIN_STORE
    lk.latent_check(_lib.latent_lib().slm_gemm(lk.C.byref(a), None, 0, -1, 0, lk._stream()), "slm_gemm")
    _close(y, want, torch.bfloat16)


# every number of slabs, rows and columns that fill no workgroup, results at an odd address; one rounding to 16 bits
@pytest.mark.parametrize("n", range(1, 9))
@pytest.mark.parametrize("rows,half", [(1, 16), (33, 96), (128, 2752)])
def test_glu_over_slabs(n, rows, half):
    from scalellm_amd import _lib
    lk = _lk()
    slabs = _rnd(3, n, rows, 2 * half)
    total = _f64(slabs).sum(0).reshape(rows, half // 16, 2, 16)
    wide = torch.full((rows, half + 5), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = wide[:, 1:1 + half]
    lk.latent_check(_lib.latent_lib().slm_glu_slabs(lk._p(out), lk._p(slabs), rows, half, n, wide.stride(0), 0.6, lk.GLU_ALPHA, lk.GLU_SHIFT,
                                                    lk._stream()), "slm_glu_slabs")
    _close(out, ref.clamped_glu(total[:, :, 0].reshape(rows, half), total[:, :, 1].reshape(rows, half), 0.6), torch.bfloat16)
    assert wide[:, 0].isnan().all() and wide[:, 1 + half:].isnan().all()


@pytest.mark.parametrize("M", [33, 64, 128])
def test_products_of_one_row_many_times(M):
    """Rows without a stride of their own (an expanded one), and rows that overlap: above 32 they are the vendor product's."""
    lk, N, K = _lk(), 192, 128
    w = _rnd(2, N, K, dtype=torch.bfloat16, std=K ** -0.5)
    layout, glu = lk.stream_layout(w), lk.stream_layout(w, glu=True)
    for x in (_rnd(1, 1, K, dtype=torch.bfloat16).expand(M, K), _rnd(1, 8 * M + K, dtype=torch.bfloat16).as_strided((M, K), (8, 1))):
        want = _f64(x) @ _f64(w).T
        _close(lk.linear(x, w, layout=layout), want, torch.bfloat16)
        out = torch.zeros(M, N // 2, dtype=torch.bfloat16, device=DEV)
        lk.linear_glu(x, w, out, 0.6, layout=glu)
        _close(out, ref.clamped_glu(want[:, :N // 2], want[:, N // 2:], 0.6), torch.bfloat16, b16=2e-2)


@pytest.mark.parametrize("M", [1, 20, 100])
def test_products_follow_weights_changed_in_place(M):
    lk, N, K = _lk(), 192, 128
    x, w = _rnd(1, M, K, dtype=torch.bfloat16), _rnd(2, N, K, dtype=torch.bfloat16, std=K ** -0.5)
    layout, glu = lk.stream_layout(w), lk.stream_layout(w, glu=True)

    def check(layout, glu):
        want, out = _f64(x) @ _f64(w).T, torch.zeros(M, N // 2, dtype=torch.bfloat16, device=DEV)
        _close(lk.linear(x, w, layout=layout), want, torch.bfloat16)
        _close(lk.linear_f32(x, w, 1.0, layout), want, torch.float32, f32=1e-5)
        _close(lk.linear_slabs(x, w, layout).t.sum(0), want, torch.float32, f32=1e-5)
        lk.linear_glu(x, w, out, 0.6, layout=glu)
        _close(out, ref.clamped_glu(want[:, :N // 2], want[:, N // 2:], 0.6), torch.bfloat16, b16=2e-2)
    check(layout, glu)
    w[N // 2:].mul_(-2.0)
    check(layout, glu)
    check(lk.stream_layout(w), lk.stream_layout(w, glu=True))
    w = w + 1.0   # (another tensor)
    check(layout, glu)


def test_streamed_weight_layout():
    lk, N, K = _lk(), 112, 192
    w = torch.arange(N * K, device=DEV).remainder(251).to(torch.bfloat16).view(N, K)
    p = torch.cat([w, w.new_zeros(16, K)])

    def order(t):   # panels of 64 rows, steps of 64 k, blocks of 16 rows, halves of 32 k, lanes (k / 8, row)
        return t.reshape(-1, 4, 16, K // 64, 2, 4, 8).permute(0, 3, 1, 4, 5, 2, 6).reshape(-1, K // 64, 4, 2, 64, 8)
    assert torch.equal(lk.stream_layout(w), order(p))
    assert torch.equal(lk.stream_layout(p, glu=True), order(p.view(2, 4, 16, K).transpose(0, 1)))
    assert lk.stream_layout(w, glu=True) is None and lk.stream_layout(w.float()) is None


def test_split_k_slabs_cover_k_once():
    lk = _lk()
    x, w = _rnd(1, 4, 8192, dtype=torch.bfloat16), _rnd(2, 64, 8192, dtype=torch.bfloat16, std=0.01)
    s = lk.linear_slabs(x, w)
    assert s.t.size(0) > 1
    _close(s.t.sum(0), _f64(x) @ _f64(w).T, torch.float32, f32=1e-5)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1, 20, 70])
def test_per_head_products_with_gate(rows, dtype):
    lk, H, K, N, head = _lk(), 3, 64, 32, 96
    x, w = _rnd(1, rows, H * head + 64, dtype=dtype), _rnd(2, H, N, K, dtype=dtype, std=0.1)
    gate = _rnd(3, rows, 16, dtype=dtype)
    out = torch.zeros(rows, H * 40, dtype=dtype, device=DEV)
    for g in (None, gate):
        lk.linear_heads(x, head, w, out, 40, gate=g)
        for h in range(H):
            want = _f64(x)[:, h * head:h * head + K] @ _f64(w)[h].T
            if g is not None:
                want = want * ref.sigmoid(_f64(gate)[:, h:h + 1])
            _close(out[:, h * 40:h * 40 + N], want, dtype)
        assert not out.view(rows, H, 40)[:, :, N:].any()


@pytest.mark.parametrize("dtype", DTYPES)
def test_clamped_glu_bends_where_it_should(dtype):
    lk, limit = _lk(), 1.25
    v = torch.tensor([-9.0, -1.5, -1.25, -1.0, -0.25, 0.0, 0.5, 1.25, 1.5, 9.0])
    g, u = torch.meshgrid(v, v, indexing="ij")
    g, u = torch.nn.functional.pad(g.reshape(4, 25), (0, 3)), torch.nn.functional.pad(u.reshape(4, 25), (0, 3))
    gu = torch.cat([g, u], dim=1).to(dtype).to(DEV)
    out = torch.empty(4, 28, dtype=dtype, device=DEV)
    lk.clamped_glu(gu, out, limit)
    _close(out, ref.clamped_glu(g.double().numpy(), u.double().numpy(), limit), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,half,pad", [(1, 8, 0), (3, 4, 0), (7, 1000, 8), (5, 1004, 0), (3, 2056, 4), (300, 264, 16)])
def test_clamped_glu_of_eights_and_fours(rows, half, pad, dtype):
    lk = _lk()
    gu = _rnd(11, rows, 2 * half + pad, dtype=dtype)
    out = torch.full((rows, half + pad), 7.0, dtype=dtype, device=DEV)
    lk.clamped_glu(gu[:, :2 * half], out[:, :half], 1.25)
    _close(out[:, :half], ref.clamped_glu(_f64(gu)[:, :half], _f64(gu)[:, half:2 * half], 1.25), dtype)
    assert (out[:, half:] == 7.0).all()


# ---- rotation, latent norm, cache --------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,q_dim,rot,rank", [(1, 32, 2, 5), (3, 64, 32, 80), (20, 96, 34, 100), (2, 32, 64, 500)])
def test_append_norms_rotates_and_writes_its_slots(heads, q_dim, rot, rank, dtype):
    from scalellm_amd.latent_layers import YarnScaling, round_up, rotary_table
    lk, eps, rows = _lk(), 1e-4, 7
    c_pad, r_pad = round_up(rank, 64), round_up(rot, 32)
    rcfg = {"base": 900.0, "dims": rot, "scaling": {"factor": 3.0, "original": 64, "fast": 8.0, "slow": 1.0}}
    cs = rotary_table(900.0, rot, 300, YarnScaling(3.0, 64, 8.0, 1.0), DEV)
    hd = q_dim + r_pad
    off_c = heads * hd
    off_r = off_c + c_pad
    proj = torch.zeros(rows, off_r + r_pad + 16, dtype=dtype, device=DEV)
    proj[:, :off_c].view(rows, heads, hd)[:, :, :q_dim + rot] = _rnd(1, rows, heads, q_dim + rot, dtype=dtype)
    proj[:, off_c:off_c + rank] = _rnd(2, rows, rank, dtype=dtype)
    proj[:, off_r:off_r + rot] = _rnd(3, rows, rot, dtype=dtype)
    before, w = _f64(proj), _rnd(4, rank)
    pos = torch.tensor([0, 1, 2, 50, 299, 64, 7], dtype=torch.int32, device=DEV)
    slots = torch.tensor([9, 3, 0, 31, 17, 4, 22], dtype=torch.int32, device=DEV)
    cache = torch.full((32, c_pad + r_pad), 5.0, dtype=dtype, device=DEV)
    q_abs = torch.full((4, heads, c_pad + r_pad), 5.0, dtype=dtype, device=DEV)
    lk.latent_append(proj, cache, q_abs, w, cs, pos, slots, heads=heads, q_dim=q_dim, q_rot=r_pad, rank=rank, c_pad=c_pad,
                     off_c=off_c, off_r=off_r, eps=eps)
    P = pos.tolist()
    rows_ = cache[slots.long()]
    _close(rows_[:, :rank], ref.rms_norm(before[:, off_c:off_c + rank], _f64(w), eps), dtype)
    _close(rows_[:, c_pad:c_pad + rot], ref.rotate(before[:, off_r:off_r + rot], P, rcfg), dtype)
    assert not rows_[:, rank:c_pad].any() and not rows_[:, c_pad + rot:].any()
    other = [i for i in range(32) if i not in slots.tolist()]
    assert (cache[other] == 5.0).all()
    q0 = before[:, :off_c].reshape(rows, heads, hd)
    q1 = proj[:, :off_c].view(rows, heads, hd)
    want = ref.rotate(q0[:, :, q_dim:q_dim + rot], P, rcfg)
    _close(q1[:, :, q_dim:q_dim + rot], want, dtype)
    assert np.array_equal(_f64(q1)[:, :, :q_dim], q0[:, :, :q_dim])
    _close(q_abs[:, :, c_pad:c_pad + rot], want[:4], dtype)
    assert not q_abs[:, :, c_pad + rot:].any() and (q_abs[:, :, :c_pad] == 5.0).all()


# rows around the tiles of the product and the largest of the one launch; more rows appended than absorbed; a query width that is
# padded for the product, and one whose rotated part a thread takes element by element: two launches
@pytest.mark.parametrize("heads,q_dim,rot,rank", [(5, 128, 64, 512), (24, 64, 16, 96), (3, 96, 32, 70), (4, 64, 12, 64)])
@pytest.mark.parametrize("rows,absorbed", [(1, 1), (5, 5), (16, 16), (33, 17), (65, 64), (256, 200), (257, 257)])
def test_append_with_absorbed_queries(heads, q_dim, rot, rank, rows, absorbed):
    """The same bits as the append and the product one after the other."""
    from scalellm_amd.latent_layers import round_up, rotary_table
    lk = _lk()
    c_pad, r_pad, k = round_up(rank, 64), round_up(rot, 32), round_up(q_dim, 64)
    cs = rotary_table(900.0, rot, 300, None, DEV)
    hd = q_dim + r_pad
    off_c = heads * hd
    proj = _rnd(1, rows, off_c + c_pad + r_pad + 16, dtype=torch.bfloat16)
    w, w_abs = _rnd(2, rank), _rnd(3, heads, c_pad, k, dtype=torch.bfloat16)
    w_abs[:, :, q_dim:] = 0
    pos = torch.arange(rows, dtype=torch.int32, device=DEV)
    slots = torch.randperm(rows, generator=torch.Generator().manual_seed(5)).int().to(DEV)
    sizes = dict(heads=heads, q_dim=q_dim, q_rot=r_pad, rank=rank, c_pad=c_pad, off_c=off_c, off_r=off_c + c_pad, eps=1e-5)
    got, want = ([proj.clone(), torch.full((rows, c_pad + r_pad), 5.0, dtype=torch.bfloat16, device=DEV),
                  torch.full((absorbed, heads, c_pad + r_pad), 5.0, dtype=torch.bfloat16, device=DEV)] for _ in range(2))
    lk.latent_append(*got, w, cs, pos, slots, **sizes, w_abs=w_abs)
    lk.latent_append(*want, w, cs, pos, slots, **sizes)
    lk.linear_heads(want[0][:absorbed], hd, w_abs, want[2].view(absorbed, -1), c_pad + r_pad)
    for g, x in zip(got, want):
        assert torch.equal(g.view(torch.int16), x.view(torch.int16))


@pytest.mark.parametrize("heads,q_dim,rot,rank", [(16, 128, 64, 512), (40, 64, 16, 250), (64, 128, 32, 128)])
@pytest.mark.parametrize("rows,absorbed", [(33, 33), (64, 64), (70, 65), (128, 127), (256, 256)])
def test_append_with_absorbed_queries_of_many_heads(heads, q_dim, rot, rank, rows, absorbed):
    test_append_with_absorbed_queries(heads, q_dim, rot, rank, rows, absorbed)


# ---- attention over the cache ------------------------------------------------------------------
class Paged:
    """Sequences of the given lengths on shuffled blocks, cache rows random (or given)."""

    def __init__(self, lens, block, c_pad, r_pad, dtype, seed=0):
        rng = np.random.default_rng(seed)
        self.lens, self.block = lens, block
        n = [(x + block - 1) // block for x in lens]
        ids = rng.permutation(sum(n) + 3)[:sum(n)]
        self.cu = np.concatenate([[0], np.cumsum(n)])
        self.table = (ids * block).astype(np.int32)
        self.cache = _rnd(seed, (sum(n) + 3) * block, c_pad + r_pad, dtype=dtype)

    def slot(self, s, p):
        return int(self.table[self.cu[s] + p // self.block]) + p % self.block

    def rows(self, s):
        return self.cache[[self.slot(s, p) for p in range(self.lens[s])]]

    def dev(self, a):
        return torch.tensor(np.asarray(a), dtype=torch.int32, device=DEV)


def _attn_ref(q, rows, p, window, scale, c_pad):
    lo = max(0, p - window + 1) if window > 0 else 0
    k = _f64(rows[lo:p + 1])
    out = []
    for h in range(q.shape[0]):
        s = k @ q[h] * scale
        e = np.exp(s - s.max())
        out.append(e / e.sum() @ k[:, :c_pad])
    return np.array(out)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("c_pad,r_pad", [(64, 32), (128, 64), (256, 32), (512, 64), (512, 32), (192, 96)])
@pytest.mark.parametrize("heads", [1, 16, 19, 40])
def test_latent_attention_sizes(c_pad, r_pad, heads, dtype):
    """Sequences of unequal lengths, rows anywhere in them, window borders, one and several splits."""
    lk = _lk()
    lens = [1, 31, 64, 65, 200, 333]
    pg = Paged(lens, 16, c_pad, r_pad, dtype, seed=heads)
    rows = [(0, 0), (1, 30), (2, 63), (3, 64), (3, 63), (4, 150), (5, 332), (5, 331), (5, 0)]
    pos = pg.dev([p for _, p in rows])
    q_cu = pg.dev(np.concatenate([[0], np.cumsum([sum(1 for s, _ in rows if s == k) for k in range(len(lens))])]))
    q = _rnd(7, len(rows), heads, c_pad + r_pad, dtype=dtype)
    scale = 2.0 * (c_pad + r_pad) ** -0.5
    for window in (0, 1, 33, 64, 200):
        want = np.stack([_attn_ref(_f64(q[i]), pg.rows(s), p, window, scale, c_pad) for i, (s, p) in enumerate(rows)])
        for kw in (dict(), dict(n_splits=1), dict(n_splits=5), dict(generic=True)):
            out = torch.full((len(rows), heads, c_pad), float("nan"), dtype=dtype, device=DEV)
            lk.latent_attention(q, pg.cache, out, pos, q_cu, pg.dev(pg.table), pg.dev(pg.cu), block_size=16, window=window,
                                scale=scale, max_kv_len=333, **kw)
            _close(out, want, dtype, f32=1e-5, b16=1.5e-2)


# The merge and the product behind it in one launch against the two: rows that leave the last workgroup of a head short, one row a workgroup and
# sixteen, splits by the rule and forced (two launches for few rows, one split, or more weights than fit), columns below, at and past a workgroup's
# 128 (then two launches, unless all workgroups are one round), with the gate and without.  The merged rows are rounded to 16 bits either way; another
# order of the splits' sums moves a rounding now and then, so 2^-8 of a few of a product's terms.
@pytest.mark.parametrize("c_pad,heads,vdim,rows,n_splits,one_launch", [
    (512, 16, 128, 9, 0, True), (512, 32, 128, 33, 0, True), (512, 32, 128, 4, 0, True), (512, 16, 128, 1, 0, False), (512, 24, 144, 100, 2, False),
    (256, 40, 96, 30, 3, True), (256, 16, 32, 33, 0, True), (128, 48, 64, 31, 5, True), (64, 17, 48, 90, 8, True), (64, 64, 16, 127, 2, True),
    (512, 128, 128, 1, 128, True), (64, 160, 32, 2, 100, True), (512, 16, 128, 40, 1, False), (64, 64, 16, 127, 40, False), (256, 127, 32, 1, 4, False),
    (512, 24, 128, 100, 2, True), (512, 32, 144, 4, 0, True), (256, 16, 256, 8, 3, True), (256, 16, 256, 9, 3, False)])
def test_latent_attention_with_its_values(c_pad, heads, vdim, rows, n_splits, one_launch):
    lk, r_pad, dt = _lk(), 64, torch.bfloat16
    lens = [40 + 53 * i % 700 for i in range(rows)]
    pg = Paged(lens, 16, c_pad, r_pad, dt)
    q = _rnd(1, rows, heads, c_pad + r_pad, dtype=dt)
    w, gate = _rnd(2, heads, vdim, c_pad, dtype=dt, std=c_pad ** -0.5), _rnd(3, rows, heads + 3, dtype=dt)
    where = (pg.dev([n - 1 for n in lens]), pg.dev(range(rows + 1)), pg.dev(pg.table), pg.dev(pg.cu))
    kw = dict(block_size=16, window=0, scale=0.1, max_kv_len=max(lens), n_splits=n_splits)
    for g in (None, gate):
        lat = torch.full((rows, heads, c_pad), float("nan"), dtype=dt, device=DEV)
        got, want = (torch.full((rows, heads * (vdim + 4) + 8), 7.0, dtype=dt, device=DEV) for _ in range(2))
        lk.latent_attention(q, pg.cache, lat, *where, values=(w, got, vdim + 4, g), **kw)
        assert (lat.isnan().all() if one_launch else not lat.isnan().any())   # (the one launch leaves no attention behind)
        lk.latent_attention(q, pg.cache, lat, *where, **kw)
        lk.linear_heads(lat.view(rows, -1), c_pad, w, want, vdim + 4, gate=g)
        _close(got, _f64(want), dt, b16=1e-2)
        assert float((got.float() - want.float()).norm() / want.float().norm()) < 2e-3
        assert (got.view(-1)[:1] != 7).all() and (got[:, heads * (vdim + 4):] == 7).all()
        assert (got[:, :heads * (vdim + 4)].view(rows, heads, vdim + 4)[:, :, vdim:] == 7).all()


# (few pairs of a row and a head, of the widest latent)
@pytest.mark.parametrize("heads,vdim,rows,n_splits,one_launch", [(16, 128, 2, 0, True), (16, 128, 7, 32, True), (32, 128, 1, 20, True), (32, 128, 1, 33, False),
                                                                 (31, 128, 1, 8, False), (32, 144, 1, 8, True)])
def test_latent_attention_of_few_rows_with_its_values(heads, vdim, rows, n_splits, one_launch):
    test_latent_attention_with_its_values(512, heads, vdim, rows, n_splits, one_launch)


@pytest.mark.parametrize("dtype", DTYPES)
def test_latent_attention_sees_exactly_its_window(dtype):
    """One key that outweighs all others: present at distance window - 1, gone at distance window."""
    lk, c_pad, r_pad, H = _lk(), 64, 32, 2
    for block in (8, 64):
        for window in (1, 2, 16, 31, 64, 65, 128, 250):
            pg = Paged([400], block, c_pad, r_pad, dtype, seed=window)
            place = 97
            big = pg.slot(0, place)
            pg.cache[:, 64] = 0
            pg.cache[big, 64], pg.cache[big, :8] = 30.0, 9.0
            at = [p for p in (place, place + 1, place + window - 1, place + window, place + window + 1) if place <= p < 400]
            q = torch.zeros(len(at), H, c_pad + r_pad, dtype=dtype, device=DEV)
            q[:, :, 64] = 1.0
            for splits in (1, 4):
                out = torch.empty(len(at), H, c_pad, dtype=dtype, device=DEV)
                lk.latent_attention(q, pg.cache, out, pg.dev(at), pg.dev([0, len(at)]), pg.dev(pg.table), pg.dev(pg.cu), block_size=block,
                                    window=window, scale=1.0, max_kv_len=400, n_splits=splits)
                for i, p in enumerate(at):
                    seen = p - place < window
                    assert (float(out[i].float()[:, :8].min()) > 8.5) == seen, (block, window, p)


@pytest.mark.parametrize("block,lens", [(1, [2500, 1023, 1024, 1025]), (2, [5000, 2049])])
def test_latent_attention_of_more_blocks_than_are_staged_at_once(block, lens):
    lk, c_pad, r_pad, H, dt = _lk(), 64, 32, 3, torch.bfloat16
    pg = Paged(lens, block, c_pad, r_pad, dt)
    q = _rnd(1, len(lens), H, c_pad + r_pad, dtype=dt)
    pos = pg.dev([n - 1 for n in lens])
    for window in (0, 1500):
        want = np.stack([_attn_ref(_f64(q[i]), pg.rows(i), n - 1, window, 0.2, c_pad) for i, n in enumerate(lens)])
        for splits in (1, 2):
            out = torch.empty(len(lens), H, c_pad, dtype=dt, device=DEV)
            lk.latent_attention(q, pg.cache, out, pos, pg.dev(range(len(lens) + 1)), pg.dev(pg.table), pg.dev(pg.cu), block_size=block,
                                window=window, scale=0.2, max_kv_len=max(lens), n_splits=splits)
            _close(out, want, dt, b16=1.5e-2)


@pytest.mark.parametrize("block", [16, 32, 128])
@pytest.mark.parametrize("c_pad,heads", [(64, 32), (128, 64), (256, 40), (512, 16), (512, 32)])
def test_latent_attention_of_whole_and_cut_tiles(c_pad, heads, block):
    """Rows that see whole tiles of 32 keys of a block, and windows that cut the first and the last of them; what is in no sequence
    is NaN and must not be read into a product."""
    lk, r_pad, dt = _lk(), 64, torch.bfloat16
    lens = [32, 63, 64, 95, 129, 300] * 4
    pg = Paged(lens, block, c_pad, r_pad, dt, seed=block)
    mine = torch.zeros(pg.cache.size(0), dtype=torch.bool)
    for s, n in enumerate(lens):
        mine[[pg.slot(s, p) for p in range(n)]] = True
    pg.cache[~mine.to(DEV)] = float("nan")
    q = _rnd(2, len(lens), heads, c_pad + r_pad, dtype=dt)
    scale = (c_pad + r_pad) ** -0.5
    for window in (0, 32, 97):
        want = np.stack([_attn_ref(_f64(q[i]), pg.rows(i), n - 1, window, scale, c_pad) for i, n in enumerate(lens)])
        for kw in (dict(), dict(n_splits=1), dict(n_splits=3)):
            out = torch.full((len(lens), heads, c_pad), float("nan"), dtype=dt, device=DEV)
            lk.latent_attention(q, pg.cache, out, pg.dev([n - 1 for n in lens]), pg.dev(range(len(lens) + 1)), pg.dev(pg.table),
                                pg.dev(pg.cu), block_size=block, window=window, scale=scale, max_kv_len=300, **kw)
            _close(out, want, dt, b16=1.5e-2)


@pytest.mark.parametrize("heads,lens", [(16, [4096] * 20 + [4000, 33, 1, 4095, 4096]), (32, [4096] * 23 + [31, 2000]), (17, [4096] * 22 + [4064, 1])])
def test_latent_attention_of_a_stream_past_the_caches(heads, lens):
    """100 MB of keys and more that one workgroup reads: loads past the caches' replacement, with splits and without, whole tiles and
    cut ones; 17 and 32 heads also as few rows of long histories, two blocks to a workgroup."""
    from scalellm_amd.decode import make_batch_inputs
    lk, c, r, block = _lk(), 512, 64, 64
    _, positions, params, n_blocks = make_batch_inputs([1] * len(lens), lens, block, DEV, seed=3)
    assert len(lens) * max(lens) * (c + r) * 2 >= 100 << 20
    q, cache = _rnd(5, len(lens), heads, c + r, dtype=torch.bfloat16), _rnd(6, n_blocks * block, c + r, dtype=torch.bfloat16)
    want = torch.empty(len(lens), heads, c, dtype=torch.float64, device=DEV)
    for i, n in enumerate(lens):
        pos = torch.arange(n, device=DEV)
        rows = cache[params.block_tables.long()[int(params.cu_block_lens[i]) + pos // block] + pos % block].double()
        want[i] = torch.softmax(q[i].double() @ rows.t() * (c + r) ** -0.5, -1) @ rows[:, :c]
    for kw in (dict(), dict(n_splits=1), dict(n_splits=3)):
        out = torch.full((len(lens), heads, c), float("nan"), dtype=torch.bfloat16, device=DEV)
        lk.latent_attention(q, cache, out, positions, params.q_cu_seq_lens, params.block_tables, params.cu_block_lens, block_size=block,
                            window=0, scale=(c + r) ** -0.5, max_kv_len=max(lens), **kw)
        # (16-bit weights and results: 2^-9 of a value each; of a row's own norm, which 4096 averaged keys leave small)
        assert ((out.double() - want).norm(dim=-1) / want.norm(dim=-1)).max() < 1.5e-2


# ---- prompt portions ---------------------------------------------------------------------------
@pytest.mark.parametrize("q_dim,r_pad,v_pad", [(32, 32, 32), (64, 32, 64), (64, 64, 128), (96, 64, 32), (128, 64, 128), (192, 64, 128)])
@pytest.mark.parametrize("window", [0, 100])
def test_portions_with_and_without_shared_tiles(q_dim, r_pad, v_pad, window):
    """Few workgroups (two groups of waves share a portion's tiles) and many (one group), at the edges of the tiles of 64
    keys (32 from 256 + 128 columns) and 128 rows, the fewest shared tiles, odd and even numbers of them."""
    from scalellm_amd.latent_layers import LatentPlan
    from scalellm_amd.layers import Portion
    lk, H, c_pad, block, dt = _lk(), 32, 64, 16, torch.bfloat16
    spans = [(1, 1), (64, 64), (65, 65), (129, 129), (5, 260), (200, 320), (31, 321), (130, 449), (400, 600), (2, 500), (3, 1000)]   # rows, context
    nb = [(k + block - 1) // block for _, k in spans]
    first = np.concatenate([[0], np.cumsum(nb)])
    cache = _rnd(3, sum(nb) * block, c_pad + r_pad, dtype=dt)
    T, dq = sum(n for n, _ in spans), q_dim + r_pad
    proj, w = _rnd(1, T, H * dq + H, dtype=dt), _rnd(2, H * (q_dim + v_pad), c_pad, dtype=dt, std=c_pad ** -0.5)
    portions, row = [], 0
    for i, (n, k) in enumerate(spans):
        portions.append(Portion(row, n, k, (np.arange(first[i], first[i + 1]) * block).astype(np.int32)))
        row += n
    got = {}
    for many in (False, True):
        out = torch.full((T, H * v_pad), float("nan"), dtype=dt, device=DEV)
        for ps in ([portions] if many else [[p] for p in portions]):   # 17 tiles of 32 heads, and up to 4
            plan = LatentPlan.build(ps, window, block, DEV)
            assert len(plan.tiles) * H > 512 if many else len(plan.tiles) * H <= 256   # (between them the contexts decide)
            ctx = lk.latent_gather(cache, plan.slots)
            kv = torch.mm(ctx[:, :c_pad], w.t())
            lk.latent_prefill(proj, ctx, kv, out, plan.tiles, heads=H, q_dim=q_dim, c_pad=c_pad, v_pad=v_pad, gate_off=H * dq,
                              window=window, scale=2 * dq ** -0.5)
        got[many] = out.double()
    for i, ((n, k), p) in enumerate(zip(spans, portions)):
        rows = cache[int(first[i]) * block:int(first[i]) * block + k]
        x, kr, pr = torch.mm(rows[:, :c_pad], w.t()).double().view(k, H, -1), rows[:, c_pad:].double(), proj[p.row0:p.row0 + n].double()
        pos, j = torch.arange(k - n, k, device=DEV)[:, None], torch.arange(k, device=DEV)[None]
        seen = (j <= pos) & (pos - j < window if window else True)
        for h in range(H):
            q = pr[:, h * dq:(h + 1) * dq]
            s = ((q[:, :q_dim] @ x[:, h, :q_dim].t() + q[:, q_dim:] @ kr.t()) * 2 * dq ** -0.5).masked_fill(~seen, -float("inf"))
            want = torch.softmax(s, 1) @ x[:, h, q_dim:] * torch.sigmoid(pr[:, H * dq + h])[:, None]
            for out in got.values():   # 16-bit weights and results: 2^-9 of each, relative to the row
                err = (out[p.row0:p.row0 + n, h * v_pad:(h + 1) * v_pad] - want).norm(dim=1)
                assert (err <= 2.0 ** -7 * want.norm(dim=1) + 2.0 ** -8).all()


@pytest.mark.parametrize("window,groups", [(0, 2), (2047, 1), (2048, 2)])
def test_portions_of_one_round(window, groups):
    """Whole prompts of 257 to 512 workgroups: windows below 2048 keys take one group of waves, whose sums come in another order.  The
    window cuts nothing here, so a call with as many heads more as take one group for certain has the same bits where this one takes one."""
    from scalellm_amd.latent_layers import LatentPlan
    from scalellm_amd.layers import Portion
    lk, c_pad, block, q_dim, r_pad, v_pad, n = _lk(), 64, 16, 128, 64, 128, 1100
    cache = _rnd(3, n + 4, c_pad + r_pad, dtype=torch.bfloat16)
    out = {}
    for H in (32, 64):   # 288 and 576 workgroups
        proj, w = (_rnd(i, *s, dtype=torch.bfloat16) for i, s in ((1, (n, 64 * 192 + 64)), (2, (64 * 256, c_pad))))
        proj, w = torch.cat([proj[:, :H * 192], proj[:, 64 * 192:]], 1), w[:H * 256] * c_pad ** -0.5
        plan = LatentPlan.build([Portion(0, n, n, np.arange(0, n, block).astype(np.int32))], window, block, DEV)
        ctx = lk.latent_gather(cache, plan.slots)
        out[H] = torch.full((n, H * v_pad), float("nan"), dtype=torch.bfloat16, device=DEV)
        lk.latent_prefill(proj, ctx, torch.mm(ctx[:, :c_pad], w.t()), out[H], plan.tiles, heads=H, q_dim=q_dim, c_pad=c_pad, v_pad=v_pad,
                          gate_off=H * 192, window=window, scale=192 ** -0.5)
    assert torch.equal(out[32], out[64][:, :32 * v_pad]) == (groups == 1)
    _close(out[32], _f64(out[64][:, :32 * v_pad]), torch.bfloat16, b16=1e-2)


@pytest.mark.parametrize("q_dim,r_pad,v_pad", [(32, 32, 32), (32, 64, 64), (64, 64, 128), (128, 32, 64), (128, 64, 128), (192, 64, 64)])
@pytest.mark.parametrize("window", [0, 1, 40, 64, 129, 300])
def test_portion_attention(q_dim, r_pad, v_pad, window):
    """Portions at several offsets of unequal sequences, with the context gathered and cut to the window by the plan."""
    from scalellm_amd.latent_layers import LatentPlan
    from scalellm_amd.layers import Portion
    lk, H, c_pad, block = _lk(), 3, 64, 16
    dt = torch.bfloat16
    spans = [(0, 140), (77, 78 + 128), (200, 217), (129, 430)]    # [start, end) of every sequence's portion
    pg = Paged([e for _, e in spans], block, c_pad, r_pad, dt)
    row0 = np.concatenate([[0], np.cumsum([e - s for s, e in spans])])
    T = int(row0[-1]) + 5
    ld = H * (q_dim + r_pad) + 16
    proj = _rnd(1, T, ld, dtype=dt)
    w = _rnd(2, H * (q_dim + v_pad), c_pad, dtype=dt, std=c_pad ** -0.5)
    portions = [Portion(int(row0[i]) + 5, e - s, e, pg.table[pg.cu[i]:pg.cu[i + 1]]) for i, (s, e) in enumerate(spans)]
    plan = LatentPlan.build(portions, window, block, DEV)
    ctx = lk.latent_gather(pg.cache, plan.slots)
    kv = torch.mm(ctx[:, :c_pad], w.t())
    out = torch.full((T, H * v_pad), float("nan"), dtype=dt, device=DEV)
    scale = 1.5 * (q_dim + r_pad) ** -0.5
    lk.latent_prefill(proj, ctx, kv, out, plan.tiles, heads=H, q_dim=q_dim, c_pad=c_pad, v_pad=v_pad,
                      gate_off=H * (q_dim + r_pad), window=window, scale=scale)
    assert torch.isnan(out[:5].float()).all()     # rows in front of the portions are not touched
    kv64 = {}
    for i, (s, e) in enumerate(spans):
        rows = pg.rows(i)
        x = _f64(torch.mm(rows[:, :c_pad], w.t())).reshape(e, H, q_dim + v_pad)
        kv64[i] = x, _f64(rows[:, c_pad:])
    want = np.zeros((T - 5, H * v_pad))
    for i, (s, e) in enumerate(spans):
        x, kr = kv64[i]
        for p in range(s, e):
            r = int(row0[i]) + p - s
            pr = _f64(proj[r + 5])
            lo = max(0, p - window + 1) if window else 0
            for h in range(H):
                q = pr[h * (q_dim + r_pad):(h + 1) * (q_dim + r_pad)]
                sc = (x[lo:p + 1, h, :q_dim] @ q[:q_dim] + kr[lo:p + 1] @ q[q_dim:]) * scale
                ex = np.exp(sc - sc.max())
                want[r, h * v_pad:(h + 1) * v_pad] = ex / ex.sum() @ x[lo:p + 1, h, q_dim:] * ref.sigmoid(pr[H * (q_dim + r_pad) + h])
    _close(out[5:], want, dt, b16=1.5e-2)
