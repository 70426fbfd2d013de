"""Products that make their few rows themselves: the same bits as the launches they replace."""
import ctypes as C

import pytest
import torch

from ht_vllm_omni_amd import _lib as L

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def gen(seed):
    return torch.Generator().manual_seed(seed)


def dev(t, dt=None):
    return t.to(device="cuda", dtype=dt or t.dtype).contiguous()


def padc(t, n):
    out = torch.zeros(*t.shape[:-1], n, dtype=t.dtype)
    out[..., :t.shape[-1]] = t
    return out


def call(fn, *a):
    """Tensors are passed as they are: the argument list keeps them alive until the kernel has run."""
    lib = L.load_decoder()
    L.check(getattr(lib, fn)(*[L.ptr(v) if isinstance(v, torch.Tensor) else v for v in a], L.current_stream()), fn, lib)
    torch.cuda.synchronize()


def filled(cls, **kw):
    s = cls()
    s.keep = kw
    for k, v in kw.items():
        setattr(s, k, L.ptr(v) if isinstance(v, torch.Tensor) else v)
    return s


def product(x, w, M, N, K, kind, one, rt, out_frag):
    n = L.load_decoder().omni_gemm_stream_splits(M, N, K) if kind == 0 and not one else 1
    out = torch.full((n, (M + 15) // 16 * 16, N), 7.0, device="cuda", dtype=torch.float32 if kind == 0 else BF)
    if isinstance(x, L.StreamRows):
        call("omni_gemm_stream_joined", C.byref(x), w, out, N, kind, one, 0.4, 0.7, C.byref(rt) if rt else None, out_frag)
    elif rt:
        call("omni_gemm_stream_rows", x, w, out, M, N, K, C.byref(rt), out_frag)
    else:
        call("omni_gemm_stream", x, w, out, M, N, K, kind, one, 0.4, 0.7, out_frag)
    return out


# what the rows come from: (kind of the product, one partial sum, table, fragment-major output), the rows' arguments
FORMS = ["shift", "embedded shift", "one sequence", "behind the sum", "plain", "final", "rows times a table", "embedded"]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("rows,width,N", [(1, 24, 32), (2, 1024, 3072), (1, 1000, 544), (3, 1024, 1056), (4, 96, 4608), (2, 1030, 2080), (2, 2048, 9216), (1, 2048, 256), (4, 640, 64)])
def test_rows_of_the_stream(form, rows, width, N):
    """Rows of one pass and of two, of one and of two pieces a thread, an end in the middle of a piece; states, zeros and rows of this batch in front; sums in one
    and in several slabs; narrow products and such as split K."""
    g, wp = gen(rows + width + N), (width + 31) // 32 * 32
    r = lambda *s, dt=torch.float32: dev(padc(torch.randn(*s, width, generator=g), wp), dt)  # noqa: E731
    V, T = 11, rows + 1
    slabs = 1 + (rows + N) % 4
    kind, one, rt, frag = 0, 0, None, 0
    ids = dev(torch.randint(-1, V, (T,), generator=g).to(torch.int32))
    src = dict(x_in=r(T), y=r(slabs, T), y_slabs=slabs, y_stride=T * wp, gain=0.7, eps=1e-5)
    shift = dict(mu=r(1, dt=BF), state=r(7), state_slot=dev(torch.tensor([3, 5, 1, 6, 2], dtype=torch.int32)), row_of_tok=dev(torch.arange(T).to(torch.int32)),
                 positions=dev(torch.tensor([9, 0, 4, 1, 2], dtype=torch.int32)[:T]))
    embedded = dict(ids=ids, table=r(V, dt=BF), vocab=V, table_scale=1.5, eps=1e-5)
    if form == "shift":
        src.update(shift)
    elif form == "embedded shift":
        src = dict(embedded, **shift)
        src["row_of_tok"] = dev(torch.tensor([0, 0, 1, 1, 1], dtype=torch.int32)[:T])
    elif form == "one sequence":
        src.update(shift, row_of_tok=dev(torch.tensor([2, 2, 2, 0, 0], dtype=torch.int32)[:T]), y_w=r(1, dt=BF))
    elif form == "behind the sum":
        src.update(post=1, alpha=1.6, y_w=r(1, dt=BF))
        kind, frag = 3, 1
    elif form == "plain":
        kind, src["y"], src["y_slabs"] = 2, r(1, T), 0      # no count of slabs is one
    elif form == "final":
        src.update(use_final=1, final_w=r(1, dt=BF), sel=dev(torch.randperm(T, generator=g).to(torch.int32)))
        one = 1
    elif form == "rows times a table":
        kind, rt = 2, filled(L.RowTable, table=dev(torch.randn(V, N, generator=g), BF), ids=ids, rows=V, ld=N)
    else:
        src = embedded
        kind, frag = 2, 1
    w = dev(torch.randn(N * wp, generator=g) * 0.1, BF)
    outs = []
    for joined in (False, True):
        x_out = None if "sel" in src else torch.full((T, wp), 5.0, device="cuda")
        a = filled(L.StreamRows, **src, rows=rows, width=width, wp=wp, elem=0, **({} if x_out is None else dict(x_out=x_out)))
        x = a
        if not joined:
            x = torch.zeros(16 * wp, device="cuda", dtype=BF)
            a.h_out, a.frag = x.data_ptr(), 1
            call("omni_stream_rows_run", C.byref(a))
        outs.append((product(x, w, rows, N, wp, kind, one, rt, frag), x_out))
    a, b = outs[0][0], outs[1][0]
    assert torch.isfinite(a.float()).all() and bool((a != 7.0).any()) and torch.equal(a, b)
    if outs[0][1] is not None:
        assert torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("q_rank,kv_rank,heads,N", [(8, 8, 1, 16), (768, 256, 16, 2048), (1536, 512, 16, 2048), (40, 72, 20, 528), (1000, 1024, 0, 64)])
@pytest.mark.parametrize("form", ["two sequences", "one sequence", "one of them live"])
def test_latents(T, q_rank, kv_rank, heads, N, form):
    """A piece a thread and three; gates and none; cache rows, gates and states too, of live rows and of a sequence's last token alone."""
    g = gen(T + q_rank + N)
    r32 = lambda n: (n + 31) // 32 * 32  # noqa: E731
    qp, rp = r32(q_rank), r32(kv_rank)
    ld, W, bs, slabs = qp + rp + r32(heads), 96, 4, 1 if form == "one sequence" else 1 + (q_rank + T) % 4
    parts = torch.zeros(slabs, T, ld)
    parts[..., :q_rank], parts[..., qp:qp + kv_rank] = torch.randn(slabs, T, q_rank, generator=g), torch.randn(slabs, T, kv_rank, generator=g)
    parts[..., qp + rp:qp + rp + heads] = torch.randn(slabs, T, heads, generator=g)
    w = dev(torch.randn(N * qp, generator=g) * 0.1, BF)
    fixed = dict(proj=dev(parts), slabs=0 if form == "one sequence" else slabs, slab_stride=T * ld, ld=ld, q_rank=q_rank, qp=qp, kv_rank=kv_rank, rp=rp, heads=max(heads, 1), qw=dev(padc(torch.randn(q_rank, generator=g), qp), BF),
                 kw=dev(padc(torch.randn(kv_rank, generator=g), rp), BF), eps=1e-6, block_table=dev(torch.tensor([[2, 0, 1], [4, 3, 5]], dtype=torch.int32)), bt_stride=3, block_size=bs,
                 row_of_tok=dev(torch.tensor([0, 0 if form == "one sequence" else 1], dtype=torch.int32)[:T]), positions=dev(torch.tensor([6, 7], dtype=torch.int32)[:T]),
                 x=dev(torch.randn(T, W, generator=g)), wp=W, state_slot=dev(torch.tensor([1, 2], dtype=torch.int32)), T=T, elem=0)
    if form == "one of them live":
        fixed["num_live"] = dev(torch.tensor([1], dtype=torch.int32))
    outs = []
    for joined in (False, True):
        own = dict(cache=torch.full((6, bs, rp), 3.0, device="cuda", dtype=BF), state=torch.full((3, W), 3.0, device="cuda"), gate=torch.full((T, max(heads, 1)), 3.0, device="cuda") if heads else None)
        out = torch.full((T, N), 7.0, device="cuda", dtype=BF)
        a = filled(L.LatentWrite, **fixed, **{k: v for k, v in own.items() if v is not None})
        if joined:
            call("omni_gemm_stream_latents", C.byref(a), w, out, N)
        else:
            cq = torch.zeros(16 * qp, device="cuda", dtype=BF)
            a.cq, a.frag = cq.data_ptr(), 1
            call("omni_latent_write_run", C.byref(a))
            call("omni_gemm_stream", cq, w, out, T, N, qp, 1, 0, 0.0, 0.0, 0)
        outs.append([out] + [v for v in own.values() if v is not None])
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    assert outs[0][0].abs().max() > 0


def values_both_ways(lens, heads, rp, n, gated, split, frag, fn="omni_latent_attn_values"):
    """The per-head product behind the attention of decode tokens, by two entries and by one."""
    g, T, bs = gen(sum(lens) + rp), len(lens), 16
    need = [(k + bs - 1) // bs for k in lens]
    bt = torch.zeros(T, max(need), dtype=torch.int32)
    for t in range(T):
        bt[t, :need[t]] = torch.arange(need[t]) * T + t
    lib = L.load_decoder()
    nb = lib.omni_latent_attn_workspace_bytes(T, heads, rp)
    w = dev(torch.randn(heads * n * rp, generator=g) * 0.1, BF)
    q, cache = dev(torch.randn(T, heads, rp, generator=g) * 0.3, BF), dev(torch.randn(max(need) * T, bs, rp, generator=g), BF)
    fixed = dict(q=q, cache=cache, block_table=dev(bt), bt_stride=bt.shape[1], block_size=bs, row_of_tok=dev(torch.arange(T).to(torch.int32)), positions=dev(torch.tensor(lens, dtype=torch.int32) - 1),
                 T=T, n_decode=T, heads=heads, rp=rp, scale=0.3, max_keys=4096, elem=0)
    if gated:
        fixed["gate"] = dev(torch.rand(T, heads, generator=g))
    outs = []
    for joined in (False, True):
        a = filled(L.LatentAttn, **fixed, out=torch.full((T, heads, rp), float("nan"), device="cuda", dtype=BF))
        if split:
            a.keep["ws"] = ws = torch.full((nb // 4,), float("nan"), device="cuda")
            a.workspace, a.workspace_bytes = ws.data_ptr(), nb
        out = torch.full(((T + 15) // 16 * 16 if frag else T, heads * n), 7.0, device="cuda", dtype=BF)
        if joined:
            call(fn, C.byref(a), w, out, n, frag)
        else:
            call("omni_latent_attn_run", C.byref(a))
            call("omni_head_gemm", a.keep["out"], w, out, T, heads, n, rp, frag)
        outs.append(out)
    return outs


@pytest.mark.parametrize("lens", [[1], [64], [65], [352], [17, 900], [2100, 60]])
@pytest.mark.parametrize("heads,rp,n,gated", [(1, 32, 32, True), (16, 256, 128, False), (16, 512, 128, True), (20, 96, 48, True)])
@pytest.mark.parametrize("split,frag", [(True, 1), (False, 0)])
def test_values_of_merged_splits(lens, heads, rp, n, gated, split, frag):
    """Rows of one split beside rows of several, and no workspace for any."""
    outs = values_both_ways(lens, heads, rp, n, gated, split, frag)
    assert torch.isfinite(outs[0].float()).all()
    close = torch.equal(*outs) if rp >= 256 else torch.allclose(outs[0].float(), outs[1].float(), rtol=2 ** -7, atol=1e-3)      # (narrower: head_gemm's waves do not split K, so one rounding to bf16 may fall the other way)
    assert close


@pytest.mark.parametrize("lens", [[40], [352], [2100, 60]])
@pytest.mark.parametrize("heads,rp,n", [(33, 64, 128), (80, 96, 64), (260, 32, 16)])
def test_values_of_more_heads_than_merge_for_themselves(lens, heads, rp, n):
    """More workgroups than compute units: the splits are merged once, the same bits at every width."""
    outs = values_both_ways(lens, heads, rp, n, True, True, 0)
    assert torch.isfinite(outs[0].float()).all() and torch.equal(*outs)


@pytest.mark.parametrize("T", [1, 3, 4, 5, 16, 17, 33, 64])
@pytest.mark.parametrize("heads,rp,n", [(16, 512, 128), (16, 256, 128), (20, 96, 48), (5, 224, 144), (3, 448, 144), (8, 32, 16), (256, 64, 16), (300, 64, 16)])
def test_products_of_merged_rows(T, heads, rp, n):
    """Rows of one split beside rows of up to 16, workgroups whose last rows are past the batch, columns that fill no second group of tiles or begin a second workgroup, more heads
    than one round takes: the bits of the attention and the product behind it, at every width."""
    lens = [(1, 64, 65, 352, 900, 2100, 17)[(5 * t) % 7] + t for t in range(T)]
    outs = values_both_ways(lens, heads, rp, n, True, True, int(heads * n % 32 == 0 and T % 2), "omni_latent_attn_products")
    assert torch.isfinite(outs[0].float()).all() and torch.equal(*outs)


def test_what_is_refused():
    lib = L.load_decoder()
    t = torch.zeros(1 << 16, device="cuda")
    p = t.data_ptr()
    for rows, wp in ((5, 1024), (3, 2048), (1, 2080), (0, 32)):
        a = L.StreamRows(x_in=p, x_out=p + 4, rows=rows, width=wp, wp=wp)
        assert lib.omni_gemm_stream_joined(C.byref(a), p, p, 32, 2, 1, 0.0, 0.0, None, 0, None) == -1, (rows, wp)
    a = L.StreamRows(x_in=p, rows=1, width=32, wp=32)
    assert lib.omni_gemm_stream_joined(C.byref(a), p, p, 40, 2, 1, 0.0, 0.0, None, 0, None) == -1
    assert lib.omni_gemm_stream_joined(C.byref(a), p, p, 32, 1, 1, 0.0, 0.0, None, 0, None) == -1
    assert lib.omni_gemm_stream_latents(C.byref(L.LatentWrite()), p, p, 32, None) == -1
    assert lib.omni_latent_attn_products(C.byref(L.LatentAttn(T=3, n_decode=2, rp=512)), p, p, 16, 0, None) == lib.omni_latent_attn_products(C.byref(L.LatentAttn(T=3, n_decode=3, rp=544)), p, p, 16, 0, None) == -1
    assert lib.omni_latent_attn_values(C.byref(L.LatentAttn(T=3, n_decode=3)), p, p, 16, 0, None) == -1
