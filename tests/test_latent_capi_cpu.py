"""C ABI of libslm_latent.so: exports match include/slm_latent.h, arguments are validated before anything is launched."""
import ctypes as C
import os
import random
import re
import subprocess

import pytest

from scalellm_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "slm_latent.h")


def _header():
    return re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)


def test_library_exports_what_the_header_declares():
    want = set(re.findall(r"SLM_API\s+[\w\s\*]+?\b(slm_\w+)\s*\(", _header()))
    out = subprocess.check_output(["nm", "-D", "--defined-only", _lib.LATENT_LIB_PATH], text=True)
    assert set(re.findall(r"\sT\s+(slm_\w+)", out)) == want
    L = _lib.latent_lib()
    assert b"gfx950" in L.slm_latent_version() and L.slm_latent_status_string(-1) == b"invalid argument"


@pytest.mark.parametrize("name,mirror", [("slm_residual_norm_args", _lib.ResidualNormArgs), ("slm_linear_args", _lib.LinearArgs),
                                         ("slm_latent_append_args", _lib.LatentAppendArgs),
                                         ("slm_latent_attn_args", _lib.LatentAttnArgs),
                                         ("slm_latent_prefill_args", _lib.LatentPrefillArgs)])
def test_ctypes_mirrors_have_the_header_layout(name, mirror):
    body = re.search(r"typedef struct %s \{(.*?)\} %s;" % (name, name), _header(), flags=re.S).group(1)
    kinds = {"int64_t": C.c_int64, "int32_t": C.c_int32, "float": C.c_float, "size_t": C.c_size_t}
    fields = []
    for decl in body.split(";"):
        decl = " ".join(decl.split()).replace("const ", "")
        if not decl:
            continue
        base, rest = decl.split(" ", 1) if "*" not in decl.split(" ")[0] else (decl.split("*")[0], "*" + decl.split("*", 1)[1])
        for v in rest.split(","):
            v = v.strip()
            ptr = "*" in v or base.endswith("*")
            fields.append((v.replace("*", "").strip(), C.c_void_p if ptr else kinds[base.rstrip("*")]))
    assert fields == list(mirror._fields_)


def test_invalid_arguments_come_back_as_status():
    L = _lib.latent_lib()
    assert L.slm_residual_norm(None, None) == -1
    a = _lib.LinearArgs()
    assert L.slm_linear(C.byref(a), None) == -1
    a.x = a.w = a.y = 4096
    a.M, a.N, a.K, a.ldx, a.ldw, a.ldy, a.batch, a.n_splits, a.dtype = 1, 16, 64, 64, 64, 16, 1, 1, _lib.SLM_BF16
    for field, bad, rc in (("K", 63, -1), ("N", 15, -1), ("ldx", 32, -1), ("dtype", 0, -2), ("ldw", 68, -5), ("n_splits", 2, -1),
                           ("epilogue", 9, -1)):
        keep = getattr(a, field)
        setattr(a, field, bad)
        assert L.slm_linear(C.byref(a), None) == rc, field
        setattr(a, field, keep)
    a.ldw = 0   # (not read by the streamed form)
    for field, bad, rc in (("K", 63, -1), ("N", 15, -1), ("ldx", 32, -1), ("ldy", 8, -1), ("dtype", _lib.SLM_F32, -2), ("ldx", 68, -5),
                           ("n_splits", 2, -1), ("batch", 2, -1), ("epilogue", _lib.LIN_GATE, -1), ("epilogue", _lib.LIN_GLU, -1), ("w", 4098, -5)):
        keep = getattr(a, field)
        setattr(a, field, bad)
        assert L.slm_linear_stream(C.byref(a), None) == rc, field
        setattr(a, field, keep)
    b = _lib.LatentAttnArgs()
    b.rows, b.batch, b.heads, b.c_pad, b.r_pad, b.block_size, b.dtype = 3, 1, 4, 64, 32, 16, _lib.SLM_BF16
    assert L.slm_latent_attn(C.byref(b), None) == -1          # null pointers
    b.block_size = 24
    assert L.slm_latent_attn(C.byref(b), None) == -1
    b.block_size, b.dtype = 16, 0
    assert L.slm_latent_attn(C.byref(b), None) == -2
    v = _lib.LinearArgs()
    assert L.slm_latent_attn_values(C.byref(b), None, None) == L.slm_latent_attn_values(C.byref(b), C.byref(v), None) == -1
    v.w, v.y, v.N, v.n_splits, v.epilogue = 4104, 4096, 64, 1, _lib.LIN_STORE
    assert L.slm_latent_attn_values(C.byref(b), C.byref(v), None) == -5
    v.w, v.epilogue = 4096, _lib.LIN_GATE
    assert L.slm_latent_attn_values(C.byref(b), C.byref(v), None) == -1   # no gate
    # what slm_linear refuses is refused in front of the attention's launch (there is no device here: a launch is another error)
    b.dtype, b.max_kv_len = _lib.SLM_BF16, 64
    b.q_abs = b.cache = b.out = b.positions = b.q_cu = b.block_table = b.block_cu = 4096
    v.x, v.epilogue, v.M, v.K, v.ldx, v.ldw, v.batch, v.dtype = 4096, _lib.LIN_STORE, 3, 64, 256, 64, 4, _lib.SLM_BF16
    for field, bad, rc in (("x", None, -1), ("K", 63, -1), ("ldx", 32, -1), ("ldw", 32, -1), ("batch", 0, -1), ("dtype", 0, -2), ("ldx", 260, -5),
                           ("x_batch", 4, -5), ("w_batch", 4, -5), ("x", 4104, -5)):
        keep = getattr(v, field)
        setattr(v, field, bad)
        assert L.slm_latent_attn_values(C.byref(b), C.byref(v), None) == rc, field
        setattr(v, field, keep)
    assert L.slm_latent_gather(None, None, None, 1, 64, None) == -1
    for args in ((None, 4096, 64, 64, 0), (4096, 4096, 72, 64, 0), (4096, 4096, 64, 72, 0), (4096, 4096, 96, 64, 1)):
        assert L.slm_stream_layout(*args, None) == -1
    assert L.slm_stream_layout(4096, 4104, 64, 64, 0, None) == -5
    assert L.slm_clamped_glu(4096, 4096, 1, 6, 12, 8, 1.0, 1.0, 1.0, _lib.SLM_BF16, None) == -1
    p = _lib.LatentPrefillArgs()
    assert L.slm_latent_prefill(C.byref(p), None) == -1
    assert L.slm_latent_prefill_supported(128, 64, 128) == 1 and L.slm_latent_prefill_supported(250, 96, 128) == 0


def test_split_plan_sizes_its_workspace():
    L = _lib.latent_lib()
    b = _lib.LatentAttnArgs()
    b.rows, b.batch, b.heads, b.c_pad, b.r_pad, b.block_size, b.dtype = 2, 2, 16, 512, 64, 64, _lib.SLM_BF16
    b.max_kv_len = 4096
    many = L.slm_latent_attn_workspace_bytes(C.byref(b))
    assert many > 0
    b.window = 64                      # a window bounds the range that can be split
    assert L.slm_latent_attn_workspace_bytes(C.byref(b)) < many
    b.window, b.rows = 0, 4096
    assert L.slm_latent_attn_workspace_bytes(C.byref(b)) == 0
    b.rows, b.dtype = 2, _lib.SLM_F32
    assert L.slm_latent_attn_workspace_bytes(C.byref(b)) == 0


@pytest.mark.parametrize("c_pad,rows,keys,blocks", [(512, 16, 4096, 1), (512, 16, 12000, 2), (512, 24, 500, 2), (512, 4, 12000, 1), (256, 8, 4096, 1),
                                                    (256, 16, 4096, 2), (128, 8, 1500, 1), (128, 16, 1500, 2), (64, 8, 4096, 1), (64, 16, 12000, 2)])
def test_head_blocks_of_few_rows_follow_the_keys(c_pad, rows, keys, blocks):
    """32 heads as two workgroups of 16 or one of both, told from the splits: 256 workgroups (512 of the narrowest latent), a tile
    of 32 keys at least each."""
    b = _lib.LatentAttnArgs()
    b.rows, b.batch, b.heads, b.c_pad, b.r_pad, b.block_size, b.dtype, b.max_kv_len = rows, rows, 32, c_pad, 64, 64, _lib.SLM_BF16, keys
    got = _lib.latent_lib().slm_latent_attn_workspace_bytes(C.byref(b)) // (rows * 32 * (c_pad + 2) * 4)
    splits = lambda n: (512 if c_pad == 64 else 256) // (rows * (2 // n))  # noqa: E731
    assert splits(1) != splits(2) and got == min(splits(blocks), (keys + 31) // 32, 64), got


def test_streamed_layout_is_made_on_the_device_of_its_weight(monkeypatch):
    """The current device may be another one while a model is built: launched there, the kernel would read foreign memory."""
    import contextlib
    import types
    import torch
    from scalellm_amd import latent_kernels as lk
    current, made_on = ["cuda:0"], []

    @contextlib.contextmanager
    def device(d):
        old, current[0] = current[0], str(d)
        yield
        current[0] = old

    def layout(*args):
        made_on.append(current[0])
        return 0
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(lk, "_stream", lambda: 0)
    monkeypatch.setattr(lk, "_p", lambda t: 4096)
    monkeypatch.setattr(lk._lib, "latent_lib", lambda: types.SimpleNamespace(slm_stream_layout=layout))
    monkeypatch.setattr(torch, "empty", lambda *a, **k: object())
    w = types.SimpleNamespace(shape=(64, 64), dtype=torch.bfloat16, is_cuda=True, is_contiguous=lambda: True, data_ptr=lambda: 4096,
                              device="cuda:3", is_inference=lambda: True)
    lk.stream_layout(w)
    assert made_on == ["cuda:3"]


def test_layouts_fit_the_memory_that_is_left(monkeypatch):
    import torch
    from scalellm_amd import latent_kernels as lk

    class Holder:
        STREAMED = (("a", "wa", False), ("b", "wb", True), ("c", "wc", False))

        def __init__(self):
            self.wa, self.wb, self.wc = (torch.zeros(n, 64, dtype=torch.bfloat16) for n in (70, 640, 64))   # 16, 80 and 8 KB laid out
    made = []
    monkeypatch.setattr(lk, "stream_layout", lambda w, glu: made.append((w.size(0), glu)) or w)

    def names(spare):
        h, made[:] = Holder(), []
        lk.lay_out([h], spare)
        return "".join(n for n in "abc" if getattr(h, n) is not None)
    assert names(None) == "abc" and made == [(70, False), (640, True), (64, False)]
    assert [names(k << 10) for k in (0, 8, 16, 24, 96, 103, 104)] == ["", "c", "a", "ac", "ab", "ab", "abc"]

    def full(w, glu):
        if w.size(0) == 640:
            raise torch.OutOfMemoryError
        return w
    monkeypatch.setattr(lk, "stream_layout", full)
    assert names(None) == "a"   # (no more after a refusal)


# one launch where K is short or the columns alone fill the chip, slabs and the GLU behind them where one workgroup would walk a long K
@pytest.mark.parametrize("N,K,M,slabs", [
    (4096, 4096, 32, 1), (512, 512, 33, 2), (1024, 1024, 64, 4), (1024, 8192, 64, 8), (4096, 768, 100, 3), (4096, 1024, 33, 2), (4096, 4096, 33, 4),
    (4096, 14336, 128, 4), (5504, 1024, 100, 1), (8192, 1536, 64, 2), (8192, 8192, 64, 2), (8192, 8192, 65, 4), (11008, 4096, 64, 1),
    (11008, 4096, 65, 2), (14336, 2048, 128, 1), (14336, 8192, 128, 2), (28672, 4096, 128, 1)])
def test_glu_products_share_a_long_contraction(N, K, M, slabs, monkeypatch):
    import types
    import torch
    from scalellm_amd import _lib as lib, latent_kernels as lk
    ran, glu = [], []
    monkeypatch.setattr(lk, "_p", lambda t: 4096)
    monkeypatch.setattr(lk, "_stream", lambda: 0)
    monkeypatch.setattr(lk, "_run_stream", lambda a: ran.append((a.epilogue, a.n_splits)))
    monkeypatch.setattr(lk._lib, "latent_lib", lambda: types.SimpleNamespace(slm_glu_slabs=lambda *a: glu.append(a[2:6]) or 0))
    t = lambda *shape: torch.empty(*shape, dtype=torch.bfloat16, device="meta")  # noqa: E731
    lk.linear_glu(t(M, K), t(N, K), t(M, N // 2), 7.0, layout=t((N + 63) // 64, K // 64, 4, 2, 64, 8))
    if slabs == 1:
        assert ran == [(lib.LIN_GLU, 1)] and not glu
    else:
        assert ran == [(lib.LIN_SLABS, slabs)] and glu == [(M, N // 2, slabs, N // 2)]


def test_glu_over_slabs_refuses_what_it_has_no_form_for():
    f = _lib.latent_lib().slm_glu_slabs
    args = lambda rows=1, half=32, n=2, ld=32, y=4096, s=4096: (y, s, rows, half, n, ld, 1.0, 1.0, 1.0, None)  # noqa: E731
    assert f(*args(rows=0)) == 0
    assert {f(*args(half=24)), f(*args(n=0)), f(*args(n=9)), f(*args(ld=31)), f(*args(y=None)), f(*args(rows=-1))} == {-1}
    assert f(*args(s=4104)) == -5


@pytest.mark.parametrize("N,K,M,slabs", [
    (512, 512, 32, 1), (512, 512, 33, 2), (512, 512, 128, 2), (2048, 896, 100, 3), (1024, 1536, 100, 6), (2048, 2048, 100, 4), (4096, 768, 65, 3),
    (4096, 1024, 65, 2), (4096, 4096, 128, 4), (4096, 14336, 128, 4), (5504, 640, 100, 1), (8192, 8192, 64, 2), (8192, 8192, 65, 4), (8192, 14336, 128, 4),
    (8192, 6144, 128, 2), (64, 32832, 1, 8)])
def test_slabs_of_streamed_products(N, K, M, slabs):
    from scalellm_amd import latent_kernels as lk
    assert lk.stream_split_count(N, K, M) == slabs


def _route(monkeypatch, product, M, N, K):
    """'stream', 'rows' or 'vendor': what serves an [M, K] x [N, K] product of weights with a streamed layout."""
    import torch
    from scalellm_amd import latent_kernels as lk
    went = []
    monkeypatch.setattr(lk, "_p", lambda t: 4096)
    monkeypatch.setattr(lk, "_run_stream", lambda a: went.append("stream"))
    monkeypatch.setattr(lk, "_run_linear", lambda a: went.append("rows"))
    monkeypatch.setattr(lk, "clamped_glu", lambda *a: None)
    monkeypatch.setattr(torch, "mm", lambda *a, **k: went.append("vendor"))
    t = lambda *shape: torch.empty(*shape, dtype=torch.bfloat16, device="meta")  # noqa: E731
    product(lk, t(M, K), t(N, K), t((N + 63) // 64, K // 64, 4, 2, 64, 8))
    return went[0]


@pytest.mark.parametrize("N,K,rows", [(6784, 4096, 32), (8128, 512, 32), (8192, 512, 64), (8192, 2048, 64), (8192, 4096, 32), (8192, 14336, 32),
                                      (9216, 4096, 64), (9216, 8192, 32), (16896, 4096, 64), (28672, 8192, 64)])
def test_stored_products_are_streamed_where_that_is_faster(N, K, rows, monkeypatch):
    for M in (1, 32, 33, 64, 65):
        assert _route(monkeypatch, lambda lk, x, w, layout: lk.linear(x, w, layout=layout), M, N, K) == ("stream" if M <= rows else "vendor"), M


def test_products_of_many_rows_are_the_vendors_where_that_is_faster():
    from scalellm_amd.latent_kernels import _tile_pays as pays
    # one row of tiles over large weights, and past it
    assert not pays(129, 28672, 4096, True) and not pays(160, 28672, 4096, False) and pays(161, 28672, 4096, True)
    assert not pays(192, 16384, 8192, True) and pays(193, 16384, 8192, True) and pays(160, 16384, 4095, True) and pays(128, 28672, 4096, True)
    # whole rounds of 256 x 256 tiles, a tile's last rows missing too; one tile more or less; short contractions and few rows; with the GLU
    assert not pays(4096, 4096, 4096, False) and not pays(3841, 4096, 2048, False) and not pays(2048, 16384, 1024, False)
    assert pays(3840, 4096, 4096, False) and pays(4097, 4096, 4096, False) and pays(4096, 4352, 4096, False)
    assert pays(4096, 4096, 960, False) and pays(1024, 16384, 4096, False) and pays(4096, 4096, 4096, True)
    # short and narrow ones are the tiles'
    assert pays(200, 512, 2048, False) and pays(129, 3664, 2048, False)


def test_products_of_changed_weights_are_slabs_as_without_a_layout():
    import torch
    from scalellm_amd import latent_kernels as lk
    layout = torch.empty(8, 64, 4, 2, 64, 8, dtype=torch.bfloat16, device="meta")
    layout.copy_of = torch.zeros(1)
    layout.copy_version = layout.copy_of._version
    assert lk.slab_rows(layout) == 128
    layout.copy_of.add_(1)
    assert lk.slab_rows(layout) == lk.slab_rows(None) == 32


def _gemm_args(M=300, N=544, K=704, epilogue=_lib.LIN_STORE):
    a = _lib.LinearArgs()
    a.x = a.w = a.y = 4096
    a.M, a.N, a.K, a.ldx, a.ldw, a.ldy, a.batch, a.n_splits, a.dtype, a.epilogue = M, N, K, K, K, N, 1, 1, _lib.SLM_BF16, epilogue
    return a


def test_tiled_products_refuse_what_they_have_no_form_for():
    L = _lib.latent_lib()
    for field, bad, rc in (("K", 63, -1), ("N", 15, -1), ("ldx", 32, -1), ("ldy", 8, -1), ("dtype", _lib.SLM_F32, -2), ("ldx", 708, -5), ("n_splits", 2, -1),
                           ("batch", 2, -1), ("epilogue", _lib.LIN_SLABS, -1), ("w", 4104, -5), ("y", 4100, -5), ("M", 1 << 22, -2)):
        a = _gemm_args()
        setattr(a, field, bad)
        assert L.slm_gemm(C.byref(a), None, 0, -1, 0, None) == rc, field
    assert L.slm_gemm(C.byref(_gemm_args()), None, 0, 7, 0, None) == -1
    assert L.slm_gemm(C.byref(_gemm_args(epilogue=_lib.LIN_GLU)), None, 0, 4, 0, None) == -2
    assert L.slm_gemm(C.byref(_gemm_args(M=0)), None, 0, -1, 0, None) == 0


def test_tiled_products_scratch_is_bounded():
    """Slabs of the cut tiles: at most one 256 x 256 tile a CU; none where nothing is cut."""
    L, rng = _lib.latent_lib(), random.Random(5)
    for _ in range(2000):
        a = _gemm_args(rng.randint(1, 9000), 32 * rng.randint(1, 1000), 64 * rng.randint(1, 250), rng.choice((_lib.LIN_STORE, _lib.LIN_GLU)))
        assert L.slm_gemm_workspace_bytes(C.byref(a), -1, 0) <= 1024 + 256 * 256 * 256 * 4
        assert L.slm_gemm_workspace_bytes(C.byref(a), -1, 1) == 0
    a = _gemm_args(2300, 4128, 320)
    assert L.slm_gemm_workspace_bytes(C.byref(a), 2, 2) == 1024 + (18 * 33 % 256) * 2 * 128 * 128 * 4
    assert L.slm_gemm_workspace_bytes(C.byref(a), 2, 4) == 1024 + (18 * 33 % 256) * 3 * 128 * 128 * 4   # five steps: no fourth slice


def test_slices_of_joined_products():
    """The rule over all sizes that it accepts: within the counters, no slice of fewer than ten steps, nothing for other rows; what the C entry takes."""
    import ctypes as C
    import random
    from scalellm_amd import _lib, latent_kernels as lk
    L, rng = _lib.latent_lib(), random.Random(5)
    for _ in range(3000):
        M, N, K = rng.randint(1, 140), 16 * rng.randint(1, 1200), 64 * rng.randint(1, 260)
        n = lk.join_count(N, K, M)
        assert 1 <= n <= 8
        a = _lib.LinearArgs()
        a.x = a.w = a.y = 1 << 20
        a.M, a.N, a.K, a.ldx, a.ldy, a.batch, a.n_splits, a.dtype = M, N, K, K, N, 1, n, _lib.SLM_BF16
        size = L.slm_linear_stream_join_bytes(C.byref(a))
        if not 16 < M <= 128 or N > 16384:
            assert n == 1 and size == 0
            assert L.slm_linear_stream_join(C.byref(a), 1 << 20, 1 << 40, 1 << 20, None) == -2
        else:
            assert size >= n * M * N * 4
            assert L.slm_linear_stream_join(C.byref(a), 1 << 20, size - 1, 1 << 20, None) < 0
            assert L.slm_linear_stream_join(C.byref(a), 1 << 20, size, None, None) < 0
        if n > 1:
            assert K // 64 // n >= 10


@pytest.mark.parametrize("M,N,K,tile,slices", [(2300, 4128, 320, 2, 2), (207, 4096, 2048, -1, 0), (300, 544, 704, 2, 3), (300, 544, 704, 2, 1)])
def test_tiled_products_scratch_in_half_precision(M, N, K, tile, slices):
    """Asked with the arguments of the call itself, the size is that of the same product in bf16; 32 bits are refused by both."""
    import ctypes as C
    from scalellm_amd import _lib
    L = _lib.latent_lib()
    a = _gemm_args(M, N, K)
    want = L.slm_gemm_workspace_bytes(C.byref(a), tile, slices)
    assert (want > 0) == (slices != 1)
    a.dtype = _lib.SLM_F16
    assert L.slm_gemm_workspace_bytes(C.byref(a), tile, slices) == want
    assert L.slm_gemm(C.byref(a), None, 0, tile, slices, None) == -2
    a.dtype = _lib.SLM_F32
    assert L.slm_gemm_workspace_bytes(C.byref(a), tile, slices) == 0
    assert L.slm_gemm_half(C.byref(a), None, 0, tile, slices, None) == -2
    assert L.slm_gemm_counted(C.byref(a), 1 << 20, 1 << 40, 1 << 20, tile, slices, None) == -2
