"""Each HIP kernel alone against a plain PyTorch float64 reference of the same op, at other sizes
than the engine tests use: odd widths, head sizes in steps of 16, groups of 1 to 16 heads, contexts
that cross pages and key chunks, a far key that must dominate, a window's edge."""
import math

import pytest
import torch

import plain_minicpm4 as P

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F64 = torch.float64


@pytest.fixture(scope="module")
def K():
    from infinilm_amd import kernels
    return kernels


def _rand(shape, seed, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def _close(got, want, tol):
    got = got.detach().cpu().to(F64)
    want = want.detach().cpu().to(F64)
    err = float((got - want).abs().max() / max(1.0, float(want.abs().max())))
    assert err < tol, f"error {err:.3e} above {tol:.1e}"


def test_constants_mirrored_in_python_equal_the_library(K):
    from infinilm_amd.csrc import lib
    L = lib.load()
    assert L.ilm_attn_tile_tokens() == K.ATT_TILE_TOKENS
    assert L.ilm_attn_mfma_step() == K.ATT_STEP
    assert L.ilm_attn_basic_chunk() == K.BASIC_CHUNK
    assert L.ilm_attn_f32_chunk() == K.F32_ATTN_CHUNK and L.ilm_attn_f32_ws_row(128) == 132
    assert L.ilm_attn_f32_tile_tokens() == K.ATT_TILE_TOKENS
    assert L.ilm_sample_host_rows() == K.SAMPLE_HOST_ROWS
    assert all(bool(L.ilm_attn_f32_tile_ok(d, 16)) == (d in K.F32_ATTN_TILE_HEADS) for d in range(16, 272, 16))
    assert L.ilm_gemm_ksplit_max_k(1) == K.KSPLIT_SPAN
    assert L.ilm_gemm_rows64_span() == K.ROWS64_SPAN


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embed(K, dtype):
    table = _rand((331, 80), 1, dtype)
    ids = torch.tensor([0, 330, 7, 7, 100], dtype=torch.int32)
    out = K.embed(ids.to(DEV), table.to(DEV), 7.5)
    assert out.dtype == torch.float32
    _close(out, table.to(F64)[ids.long()] * 7.5, 1e-6)


@pytest.mark.parametrize("dtype,wdtype,H", [(torch.float32, torch.float32, 80), (torch.bfloat16, torch.bfloat16, 331),
                                            (torch.bfloat16, torch.float32, 4096), (torch.float32, torch.float32, 1)])
def test_add_rmsnorm(K, dtype, wdtype, H):
    r = _rand((5, H), 2, scale=3.0)
    h = _rand((5, H), 3, dtype)
    w = _rand((H,), 4, wdtype) + 1
    rd = r.to(DEV).clone()
    x = K.add_rmsnorm(rd, h.to(DEV), w.to(DEV), 0.37, 1e-5, dtype)
    want_r = r.to(F64) + 0.37 * h.to(F64)
    _close(rd, want_r, 1e-6)
    want = P.plain_rmsnorm(want_r, w.to(F64), 1e-5)
    _close(x, want, 2e-6 if dtype == torch.float32 else 1e-2)
    # without a branch the residual is untouched
    rd2 = r.to(DEV).clone()
    x2 = K.add_rmsnorm(rd2, None, w.to(DEV), 1.0, 1e-5, dtype)
    assert torch.equal(rd2.cpu(), r)
    _close(x2, P.plain_rmsnorm(r.to(F64), w.to(F64), 1e-5), 2e-6 if dtype == torch.float32 else 1e-2)
    # a row's result does not depend on the batch around it
    x1 = K.add_rmsnorm(r[2:3].to(DEV).clone(), None, w.to(DEV), 1.0, 1e-5, dtype)
    assert torch.equal(x1.cpu(), x2[2:3].cpu())


@pytest.mark.parametrize("rows,H,parts,wdtype", [(64, 4096, 16, torch.bfloat16), (33, 2304, 4, torch.float32), (5, 72, 7, torch.bfloat16),
                                                 (208, 1032, 9, torch.bfloat16), (17, 4096, 3, torch.bfloat16), (40, 4104, 8, torch.bfloat16)])
def test_add_rmsnorm_of_few_rows_with_many_float_parts(K, rows, H, parts, wdtype):
    """The float32 parts of a K-split product into bfloat16 activations: 4 to 16 parts of rows up to 4096 wide take the
    kernel with 16 waves a row (3 parts, or a wider row, the general one); plain rows and fragment order; the same
    row gives the same bits whatever the rows around it."""
    r = _rand((rows, H), 2, scale=3.0)
    h = _rand((parts, rows, H), 3, scale=0.5)
    w = _rand((H,), 4, wdtype) + 1
    want_r = r.to(F64) + 0.37 * h.to(F64).sum(0)
    want = P.plain_rmsnorm(want_r, w.to(F64), 1e-5)
    rd = r.to(DEV).clone()
    x = K.add_rmsnorm(rd, h.to(DEV), w.to(DEV), 0.37, 1e-5, torch.bfloat16)
    _close(rd, want_r, 1e-6)
    _close(x, want, 1e-2)
    if rows <= K.FRAG_MAX_ROWS:
        rd2 = r.to(DEV).clone()
        xf = K.add_rmsnorm(rd2, h.to(DEV), w.to(DEV), 0.37, 1e-5, torch.bfloat16, frag=True)
        assert torch.equal(rd2, rd) and torch.equal(K.from_frag(xf), x)
        if H % 32:   # the k up to the next multiple of 32 are zeros in fragment order
            raw = xf.data.view(torch.bfloat16).view(-(-H // 32), -(-rows // 16), 4, 16, 8).cpu()
            assert not raw[-1, :, (H % 32) // 8:].any()
    one = K.add_rmsnorm(r[3:4].to(DEV).clone(), h[:, 3:4].contiguous().to(DEV), w.to(DEV), 0.37, 1e-5, torch.bfloat16)
    assert torch.equal(one, x[3:4])


@pytest.mark.parametrize("H,dtype", [(72, torch.float32), (2048, torch.float32), (2304, torch.float32), (8192, torch.bfloat16), (8192, torch.float32)])
def test_add_rmsnorm_of_any_number_of_parts(K, H, dtype):
    """One, four or eight parts are loaded at once: parts of zeros behind the others, which take the next number of slots, change no bit."""
    r, h, w = _rand((3, H), 2, scale=3.0).to(DEV), _rand((9, 3, H), 3).to(DEV), (_rand((H,), 4, dtype) + 1).to(DEV)
    for parts in (1, 2, 3, 4, 5, 8, 9):
        got = []
        for total in {parts, 4 if parts <= 4 else 8, 9, 16}:
            padded = torch.zeros((max(total, parts), 3, H), device=DEV)
            padded[:parts] = h[:parts]
            rd = r.clone()
            got.append((K.add_rmsnorm(rd, padded, w, 0.37, 1e-5, dtype), rd))
        assert all(torch.equal(x, got[0][0]) and torch.equal(rd, got[0][1]) for x, rd in got)
        want = r.to(F64) + 0.37 * h[:parts].to(F64).sum(0)
        _close(got[0][1], want, 1e-6)
        _close(got[0][0], P.plain_rmsnorm(want, w.to(F64), 1e-5), 2e-6 if dtype == torch.float32 else 1e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,d,rd,page", [(4, 2, 16, 16, 4), (3, 1, 48, 48, 16), (5, 5, 32, 16, 8), (2, 1, 80, 0, 16)])
def test_rope_and_cache_write(K, dtype, nh, nkv, d, rd, page):
    T, max_pos = 9, 50
    qkv = _rand((T, (nh + 2 * nkv) * d), 5, dtype)
    pos = torch.tensor([0, 1, 2, 17, 49, 3, 3, 30, 11], dtype=torch.int32)
    cfg = {"hidden_size": d, "num_attention_heads": 1, "max_position_embeddings": max_pos, "rope_theta": 777.0,
           "partial_rotary_factor": rd / d if 0 < rd < d else 1.0}
    if rd > 0:
        cos, sin = P.plain_rope_tables(cfg)
    else:
        cos, sin = torch.zeros(max_pos, 0, dtype=F64), torch.zeros(max_pos, 0, dtype=F64)
    n_pages = 7
    kc = torch.zeros((n_pages, nkv, page, d), dtype=dtype, device=DEV)
    vc = torch.zeros((n_pages, nkv, d, page), dtype=dtype, device=DEV)
    slots = torch.tensor([5 * page + 1, 0, 2 * page + page - 1, -1, 6 * page, 3 * page + 2, page, page + 1, 4 * page],
                         dtype=torch.int32)
    buf = qkv.to(DEV).clone()
    K.rope_kvwrite(buf, pos.to(DEV), cos.float().to(DEV), sin.float().to(DEV), kc, vc, slots.to(DEV), nh, nkv, d, rd)
    x = qkv.to(F64).view(T, nh + 2 * nkv, d)
    want_q = P.plain_apply_rope(x[:, :nh], pos, cos, sin, rd) if rd else x[:, :nh]
    want_k = P.plain_apply_rope(x[:, nh:nh + nkv], pos, cos, sin, rd) if rd else x[:, nh:nh + nkv]
    tol = 2e-6 if dtype == torch.float32 else 1e-2
    got = buf.cpu().view(T, nh + 2 * nkv, d)
    _close(got[:, :nh], want_q, tol)
    _close(got[:, nh:nh + nkv], want_k, tol)
    assert torch.equal(got[:, nh + nkv:], qkv.view(T, nh + 2 * nkv, d)[:, nh + nkv:])   # v untouched
    for t in range(T):
        s = int(slots[t])
        if s < 0:
            continue
        pg, off = s // page, s % page
        assert torch.equal(kc[pg, :, off, :].cpu(), got[t, nh:nh + nkv])        # the rotated key is what is cached
        assert torch.equal(vc[pg, :, :, off].cpu(), got[t, nh + nkv:])           # values lie transposed
    written = {int(s) for s in slots if s >= 0}
    mask = torch.ones(n_pages * page, dtype=torch.bool)
    mask[list(written)] = False
    assert not kc.cpu().permute(0, 2, 1, 3).reshape(n_pages * page, -1)[mask].any()  # nothing else was touched


@pytest.mark.parametrize("M,nh,nkv,d,Kd,page,bias", [(5, 4, 2, 32, 96, 8, False), (16, 32, 2, 128, 4096, 64, False),
                                                     (1, 3, 3, 64, 200, 16, True), (8, 16, 2, 64, 1024, 16, False),
                                                     (3, 2, 1, 96, 8192, 4, True), (17, 4, 2, 32, 96, 8, True),
                                                     (32, 32, 2, 128, 4096, 64, False), (24, 16, 2, 64, 1024, 16, False),
                                                     (29, 3, 3, 96, 2056, 16, True)])
def test_projection_with_rotation_and_cache_write_in_one_kernel(K, M, nh, nkv, d, Kd, page, bias):
    """The decode-side fused kernel against the plain product + rotation, and against the
    product kernel followed by the rotation kernel."""
    max_pos = 300
    N = (nh + 2 * nkv) * d
    x, w = _rand((M, Kd), 21, torch.bfloat16), _rand((N, Kd), 22, torch.bfloat16, scale=Kd ** -0.5)
    b = _rand((N,), 23, torch.bfloat16) if bias else None
    g = torch.Generator().manual_seed(24)
    pos = torch.randint(0, max_pos, (M,), generator=g, dtype=torch.int32)
    pos[0] = max_pos - 1
    cfg = {"hidden_size": d, "num_attention_heads": 1, "max_position_embeddings": max_pos, "rope_theta": 5000.0}
    cos, sin = P.plain_rope_tables(cfg)
    n_pages = M + 2
    slots = (torch.randperm(n_pages, generator=g)[:M] * page + torch.randint(0, page, (M,), generator=g)).to(torch.int32)
    if M > 2:
        slots[2] = -1   # a token that is not cached
    dev = lambda t: None if t is None else t.to(DEV)
    caches = []
    for fused in (True, False):
        kc = torch.zeros((n_pages, nkv, page, d), dtype=torch.bfloat16, device=DEV)
        vc = torch.zeros((n_pages, nkv, d, page), dtype=torch.bfloat16, device=DEV)
        if fused:
            q = K.qkv_rope_gemm(dev(x), dev(w), dev(b), dev(pos), dev(cos.float()), dev(sin.float()), kc, vc, dev(slots),
                                nh, nkv, d, d)
            assert q is not None
        else:
            qkv = K.gemm(dev(x), dev(w), dev(b))
            K.rope_kvwrite(qkv, dev(pos), dev(cos.float()), dev(sin.float()), kc, vc, dev(slots), nh, nkv, d, d)
            q = qkv[:, :nh * d]
        caches.append((q.cpu().float(), kc.cpu().float(), vc.cpu().float()))
    y = P.plain_linear(x.to(F64), w.to(F64), None if b is None else b.to(F64)).view(M, nh + 2 * nkv, d)
    want_q = P.plain_apply_rope(y[:, :nh], pos, cos, sin, d).reshape(M, nh * d)
    want_k = P.plain_apply_rope(y[:, nh:nh + nkv], pos, cos, sin, d)
    q, kc, vc = caches[0]
    _close(q, want_q, 1e-2)
    for t in range(M):
        s = int(slots[t])
        if s < 0:
            continue
        _close(kc[s // page, :, s % page, :], want_k[t], 1e-2)
        _close(vc[s // page, :, :, s % page], y[t, nh + nkv:], 1e-2)
    # the two paths round the projection to bfloat16 at the same place: they agree to an ulp of the result
    for a, b_ in zip(caches[0], caches[1]):
        assert (a - b_).abs().max() <= 2 ** -7 * max(a.abs().max(), 1e-6)
        assert ((a != 0) == (b_ != 0)).all()   # and write the same places, nothing else


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_swiglu_and_gather(K, dtype):
    gu = _rand((7, 2 * 200), 6, dtype, 2.0)
    out = K.swiglu(gu.to(DEV))
    g, u = gu.to(F64)[:, :200], gu.to(F64)[:, 200:]
    _close(out, P.plain_swiglu(g, u), 2e-6 if dtype == torch.float32 else 1e-2)
    x = _rand((11, 96), 7, dtype)
    idx = torch.tensor([10, 0, 3, 3], dtype=torch.int32)
    assert torch.equal(K.gather_rows(x.to(DEV), idx.to(DEV)).cpu(), x[idx.long()])


@pytest.mark.parametrize("parts,T,H", [(2, 5, 96), (4, 16, 1000), (1, 3, 7)])
def test_gather_of_parts_is_one_launch(K, monkeypatch, parts, T, H):
    """A stream whose branch is due in the parts of a K-split product: the rows of all parts at once."""
    from infinilm_amd.parts.base import ResidualStream

    x, r = _rand((parts, T, H), 8).to(DEV), _rand((T, H), 9).to(DEV)
    idx = torch.tensor([T - 1, 0, T - 1], dtype=torch.int32, device=DEV)
    stream = ResidualStream(r)
    stream.push(x, 1.0)
    calls, run = [], K._run
    monkeypatch.setattr(K, "_run", lambda name, *a: (calls.append(name), run(name, *a))[1])
    last = stream.gather(idx)
    assert calls == ["ilm_gather_rows"] * 2
    assert torch.equal(last.residual, r[idx.long()]) and torch.equal(last.pending, x[:, idx.long()])
    wide = _rand((parts, T + 2, H), 10).to(DEV)[:, :T]      # parts further apart than their rows
    assert torch.equal(K.gather_rows(wide, idx), wide[:, idx.long()])


@pytest.mark.parametrize("M,N,K_", [(1, 1, 1), (5, 331, 80), (64, 96, 200), (130, 70, 33), (3, 4608, 4096), (17, 331, 4100),
                                    (33, 50, 12296), (48, 4608, 1032), (8, 16400, 64), (20, 32768, 256), (200, 96, 200),
                                    (65, 130, 4), (300, 1100, 1028), (129, 257, 44), (2048, 1024, 4096)])
def test_gemm_float32_is_true_float32(K, M, N, K_):
    a, w, b = _rand((M, K_), 8), _rand((N, K_), 9), _rand((N,), 10)
    out = K.gemm(a.to(DEV), w.to(DEV), b.to(DEV), 0.25)
    want = P.plain_linear(a.to(F64), w.to(F64), b.to(F64), 0.25)
    _close(out, want, 2e-6 * math.sqrt(K_))   # no reduced-precision matrix mode: errors of float32 sums only
    # Rows do not depend on the batch around them, bit for bit: the few-rows kernel (up to 64 rows) and the tile
    # kernel (more) sum every output in one order, fixed by K alone (as does the plain ascending-k kernel, which
    # takes every row count of a K that is no multiple of 4).
    one = K.gemm(a[M // 2:M // 2 + 1].to(DEV), w.to(DEV), b.to(DEV), 0.25)
    assert torch.equal(one.cpu(), out[M // 2:M // 2 + 1].cpu())
    some = K.gemm(a[:min(M, 3)].to(DEV), w.to(DEV), b.to(DEV), 0.25)
    assert torch.equal(some.cpu(), out[:min(M, 3)].cpu())
    more = K.gemm(torch.cat([a, a[:70]]).to(DEV), w.to(DEV), b.to(DEV), 0.25)
    assert torch.equal(more[:M].cpu(), out.cpu())


@pytest.mark.parametrize("M,I,K_,bias,act", [(1, 15, 36, False, "silu"), (8, 4100, 260, True, "gelu_tanh"), (16, 33, 1028, False, "silu"),
                                             (33, 100, 64, True, "silu"), (64, 5760, 96, False, "gelu_tanh")])
def test_gemm_float32_with_the_activation_in_its_epilogue(K, M, I, K_, bias, act):
    """Bit for bit the projection and the activation kernel one after the other, at the edges of tiles and row groups."""
    x, w = _rand((M, K_), 70).to(DEV), _rand((2 * I, K_), 71, scale=0.1).to(DEV)
    b = _rand((2 * I,), 72).to(DEV) if bias else None
    got = K.gateup_glu_f32(x, w, b, act=act)
    assert torch.equal(got, K.swiglu(K.gemm(x, w, b), act))


@pytest.mark.parametrize("M,nh,nkv,d,page,K_,bias", [(1, 4, 2, 32, 4, 64, False), (9, 3, 3, 64, 64, 132, True), (17, 6, 1, 128, 16, 1028, False),
                                                     (40, 2, 2, 96, 8, 36, True), (64, 36, 36, 64, 64, 96, False)])
def test_gemm_float32_with_the_rotation_in_its_epilogue(K, M, nh, nkv, d, page, K_, bias):
    """Bit for bit the projection and the kernel that rotates and writes the cache; a row without a slot writes nothing."""
    x, w = _rand((M, K_), 73).to(DEV), _rand(((nh + 2 * nkv) * d, K_), 74, scale=0.1).to(DEV)
    b = _rand(((nh + 2 * nkv) * d,), 75).to(DEV) if bias else None
    g = torch.Generator().manual_seed(M)
    pos = torch.randint(0, 500, (M,), generator=g, dtype=torch.int32).to(DEV)
    ang = torch.rand((500, d // 2), generator=g) * 6.28
    cos, sin = torch.cos(ang).to(DEV), torch.sin(ang).to(DEV)
    pages = -(-M // page) + 1
    slots = torch.randperm(pages * page, generator=g)[:M].to(torch.int32)
    slots[M // 2] = -1
    slots = slots.to(DEV)
    caches = [[torch.zeros((pages, nkv, page, d), device=DEV), torch.zeros((pages, nkv, d, page), device=DEV)] for _ in range(2)]
    got = K.qkv_rope_f32(x, w, b, pos, cos, sin, *caches[0], slots, nh, nkv, d, d)
    rows = K.gemm(x, w, b)
    K.rope_kvwrite(rows, pos, cos, sin, *caches[1], slots, nh, nkv, d, d)
    assert torch.equal(got, rows[:, :nh * d])
    assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])
    assert K.qkv_rope_f32(x, w, b, pos, cos, sin, None, None, None, nh, nkv, d, d).equal(got)


@pytest.mark.parametrize("M,N,K_", [(1, 1024, 1032), (16, 1000, 2048), (3, 2305, 2056), (16, 40, 3080), (9, 5000, 4096), (2, 300, 4096)])
def test_gemm_few_rows_in_short_parts(K, M, N, K_):
    """Up to 16 rows on their way into a residual sum, K in parts of 1,024: parts that do not fill up, more tiles than
    workgroups.  bfloat16 operands are exact in float64, the parts' sum is float: 2^-24 a sum of K products."""
    a, w = _rand((M, K_), 50, torch.bfloat16), _rand((N, K_), 51, torch.bfloat16)
    parts = K.gemm(a.to(DEV), w.to(DEV), allow_parts=True)
    assert parts.dtype == torch.float32 and parts.shape == (-(-K_ // K.KSPLIT_FEW_SPAN), M, N)
    _close(parts.sum(0), P.plain_linear(a.to(F64), w.to(F64)), 2e-6 * math.sqrt(K_))
    one = K.gemm(a[M - 1:].to(DEV), w.to(DEV), allow_parts=True)
    assert torch.equal(one[:, 0], parts[:, M - 1])      # a row's bits do not depend on the rows around it


@pytest.mark.parametrize("M,N,K_", [(1, 15, 4), (8, 4097, 36), (9, 33, 1028), (17, 16385, 68), (40, 260, 260), (64, 257, 4096), (65, 63, 8),
                                    (127, 129, 2052), (129, 257, 1024), (192, 4100, 516), (333, 640, 8192)])
def test_gemm_float32_in_pieces(K, M, N, K_):
    """The products in three bfloat16 pieces a float, at the edges of their tiles, rows and slices: every tile gives the same bits, and
    the error against float64 stays below that of sums of floats rounded every four k, 2.1e-7 sqrt(K / 1024) of the norm
    (measured with the float matrix instruction at K 1024, 4096 and 16,384), here with operands over six decades and
    with the largest numbers of the type."""
    from infinilm_amd.csrc import lib
    g = torch.Generator().manual_seed(M * 7 + N)
    a, w = torch.randn((M, K_), generator=g), torch.randn((N, K_), generator=g)
    a *= torch.exp(1.5 * torch.randn((M, K_), generator=g))
    a[0] *= 1e30
    a[M // 2, K_ - 1] = 3.4028234663852886e38
    w[:, K_ - 1] *= 1e-30
    ad, wd = a.to(DEV), w.to(DEV)
    out = K.gemm(ad, wd)
    want = ad.to(F64) @ wd.to(F64).T
    rel = ((out.to(F64) - want).norm(dim=1) / want.norm(dim=1)).max()
    assert float(rel) < 2.1e-7 * math.sqrt(max(K_, 1024) / 1024)
    for tile in (1, 2, 3):
        c = torch.full_like(out, float("nan"))
        assert lib.load().ilm_gemm_f32_tile(c.data_ptr(), ad.data_ptr(), wd.data_ptr(), None, M, N, K_, K_, K_, N, 1.0, tile,
                                            torch.cuda.current_stream().cuda_stream) == 0
        assert torch.equal(c, out), f"tile {tile}"


@pytest.mark.parametrize("M,N,K_", [(65, 63, 36), (127, 257, 68), (129, 1030, 260), (300, 513, 1028), (130, 255, 2052), (200, 301, 8192), (1100, 8200, 132)])
@pytest.mark.parametrize("odd", [False, True])
def test_gemm_float32_cut_tiles_give_the_same_bits(K, M, N, K_, odd):
    """Tiles whose slices of K go to several workgroups, as many as there are slices and fewer, few slices and eight, alone and after a round of whole
    tiles, with a bias, a factor and rows that cannot be stored four at a time; infinities, NaNs and sums that the pieces cannot give among them."""
    from infinilm_amd.csrc import lib
    L = lib.load()
    g = torch.Generator().manual_seed(M + N + odd)
    a, w, bias = torch.randn((M, K_), generator=g), torch.randn((N, K_), generator=g), torch.randn((N,), generator=g)
    if odd:
        a[M // 3, 3], a[M // 2, K_ - 1], a[M - 1] = math.inf, math.nan, a[M - 1] * 2.0 ** -80
        w[N // 2, 5], w[N - 1, :2], a[0, :2] = -math.inf, torch.tensor([3e38, -3e38]), torch.tensor([3.0, 3.0])
    a, w, bias = a.to(DEV), w.to(DEV), bias.to(DEV)
    steps = -(-K_ // 32)
    slices = -(-steps // (-(-steps // 8)))
    ld = N + (3 if odd else 0)
    args = (a.data_ptr(), w.data_ptr(), bias.data_ptr(), M, N, K_, K_, K_, ld, 0.5)
    ws = torch.empty(((-(-M // 128)) * (-(-N // 256)) * slices * 128 * 256,), device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    want = torch.full((M, ld), 7.0, device=DEV)
    assert L.ilm_gemm_f32_tile(want.data_ptr(), *args, 1, stream) == 0
    assert not odd or not torch.isfinite(want).all()
    for parts in sorted({0, 1, 2, min(3, slices), slices}):
        c = torch.full((M, ld), 7.0, device=DEV)
        assert L.ilm_gemm_f32_cut(c.data_ptr(), *args, parts, ws.data_ptr(), ws.numel(), stream) == 0
        _same(c, want)
    assert L.ilm_gemm_f32_cut(c.data_ptr(), *args, slices + 1, ws.data_ptr(), ws.numel(), stream) != 0
    assert L.ilm_gemm_f32_cut(c.data_ptr(), *args, 0, ws.data_ptr(), 100, stream) != 0


@pytest.mark.parametrize("M", [1, 40, 130])
@pytest.mark.parametrize("K_", [4, 32, 1028, 4096])
def test_gemm_float32_operands_of_one_mantissa(K, M, K_):
    """What is left out of a product has one sign where all operands are alike, and does not average out.  It is at most 2^-24 of
    it; the sum of a step of 32 k is rounded once (2^-24 at most) and its small products before that (far less: half of that
    is allowed), and equal addends round the same way in every step of a slice, of which there are K / 256.  All-positive operands of any mantissa: no error of one sign (a tenth of 2^-24 over 10,000 outputs)."""
    N = 260
    same = [0x3F80FF80, 0x3F807FC0, 0x3F817F40, 0x3FFFFFFF, 0x3F800001, 0x3FAAAAAB]      # (the first two: the largest losses with h cut off and rounded)
    for x in same:
        for w in same:
            pair = torch.tensor([x, w], dtype=torch.int32).view(torch.float32)
            a, b = pair[0].expand(M, K_).contiguous().to(DEV), pair[1].expand(N, K_).contiguous().to(DEV)
            want = K_ * float(pair[0]) * float(pair[1])
            assert abs(K.gemm(a, b).to(F64) / want - 1).max() < 2.0 ** -24 * (2.5 + K_ / 256), (hex(x), hex(w))
    g = torch.Generator().manual_seed(K_ + M)
    a, b = (1 + torch.rand((M, K_), generator=g)).to(DEV), (1 + torch.rand((10000 // M + 1, K_), generator=g)).to(DEV)
    want = a.to(F64) @ b.to(F64).T
    assert abs((K.gemm(a, b).to(F64) / want - 1).mean()) < 2.0 ** -24 / 10


def _same(a, b):
    torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("M,N,K_", [(1, 17, 36), (8, 40, 132), (33, 64, 260), (64, 33, 4), (150, 270, 68)])
def test_gemm_float32_infinities(K, M, N, K_):
    """Infinities, NaNs, the largest numbers and sums that leave the floats' range on the way: what float arithmetic has for them, the
    same bits from every kernel.  All other numbers are small and whole, so sums are exact, or beside a large number good to its
    last bits, and float64's is the answer."""
    from infinilm_amd.csrc import lib
    inf, big = math.inf, 3.4028234663852886e38
    g = torch.Generator().manual_seed(M + N)
    a = torch.randint(-9, 10, (M, K_), generator=g).float()
    w = torch.randint(-9, 10, (2 * N, K_), generator=g).float()
    for i, v in enumerate((inf, -inf, math.nan, big, -big, inf, 2.0)):
        a[i % M, (5 * i) % K_] = v
    for i, v in enumerate((0.0, -inf, 2.0 ** 125, math.nan)):     # (2^125: what it cancels with a multiple of the largest number is no small sum)
        w[(3 * i) % N, (5 * i) % K_] = v
    w[N - 1] = 0.0
    w[N - 1, :2], a[M // 2, :2] = torch.tensor([big, -big]), torch.tensor([3.0, 3.0])
    want = (a.to(F64)[:, None, :] * w.to(F64)[None]).sum(-1).float()
    assert not torch.isfinite(want).all() and (torch.isfinite(want).any() or M == 1)
    ad, wd = a.to(DEV), w.to(DEV)
    out = K.gemm(ad, wd)
    torch.testing.assert_close(out.cpu(), want, rtol=2.0 ** -22, atol=0, equal_nan=True)
    for tile in (1, 2, 3):
        c = torch.full_like(out, 7.0)
        assert lib.load().ilm_gemm_f32_tile(c.data_ptr(), ad.data_ptr(), wd.data_ptr(), None, M, 2 * N, K_, K_, K_, 2 * N, 1.0, tile,
                                            torch.cuda.current_stream().cuda_stream) == 0
        _same(c, out)
    if M <= 64:
        _same(K.gateup_glu_f32(ad, wd, None), K.swiglu(out))


@pytest.mark.parametrize("M,N,K_", [(1, 17, 64), (40, 33, 1028), (130, 270, 68)])
@pytest.mark.parametrize("e", [-64, -108, -112, -119, -126, -130])
def test_gemm_float32_tiny_operands(K, M, N, K_, e):
    """Operands around the floats' smallest normal number and some way below: as good as others.  All products are positive, so a sum in
    floats of at most 1,028 of them, pieces or not, is good to 2^-24 sqrt(K) of itself at worst."""
    g = torch.Generator().manual_seed(M - e)
    a, w = (1.0 + torch.rand((M, K_), generator=g)) * 2.0 ** e, (1.0 + torch.rand((N, K_), generator=g)) * 2.0 ** 31
    a, w = a.to(DEV), w.to(DEV)
    want = a.to(F64) @ w.to(F64).T
    rel = ((K.gemm(a, w).to(F64) - want) / want).abs().max()
    assert float(rel) < 2.0 ** -24 * math.sqrt(K_)


@pytest.mark.parametrize("M,N,K_,out_dtype", [
    (1, 16, 32, torch.bfloat16), (1, 4608, 4096, torch.bfloat16), (8, 331, 80, torch.float32), (17, 96, 200, torch.bfloat16),
    (33, 200, 96, torch.bfloat16), (64, 73448, 128, torch.float32), (48, 100, 2048, torch.bfloat16),
    (7, 50, 100, torch.bfloat16),        # K no multiple of 8: the plain kernel takes it
    (100, 176, 80, torch.bfloat16), (300, 512, 256, torch.bfloat16), (65, 40, 64, torch.float32), (40, 331, 96, torch.float32),
    (32, 4608, 4096, torch.bfloat16), (25, 331, 4096, torch.float32), (20, 100, 1032, torch.bfloat16),   # two row groups in registers
    (31, 50, 4104, torch.bfloat16),      # K beyond what two row groups hold: the library
])
def test_gemm_bfloat16(K, M, N, K_, out_dtype):
    a, w = _rand((M, K_), 11, torch.bfloat16), _rand((N, K_), 12, torch.bfloat16)
    alpha = 0.3 if out_dtype == torch.float32 else 1.0
    out = K.gemm(a.to(DEV), w.to(DEV), None, alpha, out_dtype)
    assert out.dtype == out_dtype
    want = P.plain_linear(a.to(F64), w.to(F64), None, alpha)
    _close(out, want, 1e-5 if out_dtype == torch.float32 else 6e-3)
    if M <= 64:
        b = _rand((N,), 13, torch.bfloat16)
        out = K.gemm(a.to(DEV), w.to(DEV), b.to(DEV), 0.5, out_dtype)
        _close(out, P.plain_linear(a.to(F64), w.to(F64), b.to(F64), 0.5), 1e-5 if out_dtype == torch.float32 else 6e-3)


@pytest.mark.parametrize("M,N,K_", [(8, 4096, 16384), (1, 50, 8200), (16, 331, 12296), (17, 4096, 4096), (64, 4096, 16384),
                                    (48, 331, 200), (35, 50, 8200), (128, 1030, 1096), (97, 64, 72), (32, 4096, 16384),
                                    (20, 331, 12296), (27, 50, 8200), (5, 96, 5760), (30, 2304, 5760), (192, 4096, 16384), (208, 331, 4096),
                                    (150, 331, 1096), (177, 96, 200)])
@pytest.mark.parametrize("tall", [True, False])
def test_gemm_split_over_k_and_its_consumer(K, monkeypatch, M, N, K_, tall):
    """Few rows and long K: the product comes as float32 parts; add_rmsnorm sums them in order.  `tall`: with the
    product that keeps chunks of X in LDS (17 to 208 rows of a matrix that fills the chip), and with the kernels
    that serve when it is switched off."""
    monkeypatch.setattr(K, "USE_TALL", tall)
    a, w = _rand((M, K_), 14, torch.bfloat16), _rand((N, K_), 15, torch.bfloat16, 0.05)
    if M > 64 and not (tall and K._tall_fills_the_chip(N, K_, torch.device(DEV))):
        # many rows of a small matrix (or without that product) are left to the library on the engine's path
        assert K.gemm(a.to(DEV), w.to(DEV), allow_parts=True).dtype == torch.bfloat16
        if not tall:
            return
        monkeypatch.setattr(K, "TALL_MIN_WGS_PER_CU", -1.0)   # the kernel is tested all the same
    parts = K.gemm(a.to(DEV), w.to(DEV), allow_parts=True)
    if tall and 16 < M <= K.TALL_MAX_ROWS and K_ % 8 == 0 and K._tall_fills_the_chip(N, K_, torch.device(DEV)):
        assert parts.shape[0] == K._tall_plan(M, N, K_)[1] <= K.TALL_MAX_PARTS
    elif 16 < M <= 64 and K_ % 8 == 0:   # K ranges of 1024 (up to 32 rows with K beyond 4096: ranges of 4096)
        assert parts.shape[0] == (-(-K_ // 4096) if M <= 32 and K_ > 4096 else -(-K_ // 1024))
    if parts.dim() == 2:   # short K and few rows: one float32 result
        assert K_ <= 4096 and M <= 16
        parts = parts[None]
    assert parts.dim() == 3 and parts.dtype == torch.float32
    assert M > 16 or K_ <= 4096 or parts.shape[0] == -(-K_ // 4096)   # up to 16 rows: K ranges of 4096
    want = P.plain_linear(a.to(F64), w.to(F64))
    _close(parts.sum(0), want, 1e-5)
    whole = K.gemm(a.to(DEV), w.to(DEV))
    assert whole.dim() == 2 and whole.dtype == torch.bfloat16
    short = K.gemm(a[:, :256].contiguous().to(DEV), w[:, :256].contiguous().to(DEV), allow_parts=True)
    # short K: float32, not rounded to bfloat16 (more than 16 rows: parts)
    # (many rows of a small matrix: the library's bfloat16 result)
    assert (short.dtype == torch.float32 and short.dim() == 2) if M <= 16 else (short.dim() == 3 or M > 64)
    _close(whole, want, 6e-3)
    r = _rand((M, N), 16, scale=2.0)
    nw = _rand((N,), 17, torch.bfloat16) + 1
    rd = r.to(DEV).clone()
    x = K.add_rmsnorm(rd, parts, nw.to(DEV), 0.3, 1e-6, torch.bfloat16)
    want_r = r.to(F64) + 0.3 * want
    _close(rd, want_r, 1e-5)
    _close(x, P.plain_rmsnorm(want_r, nw.to(F64), 1e-6), 1e-2)


@pytest.mark.parametrize("M,I,N", [(8, 16384, 4096), (3, 200, 96), (16, 4104, 50), (17, 4104, 50), (32, 16384, 4096),
                                   (24, 200, 96), (33, 96, 331)])
def test_swiglu_inside_the_down_projection(K, M, I, N):
    gu = _rand((M, 2 * I), 18, torch.bfloat16, 1.5)
    w = _rand((N, I), 19, torch.bfloat16, 0.05)
    if M > 32:   # more rows: the activation kernel and a product of its own
        assert K.swiglu_gemm(gu.to(DEV), w.to(DEV)) is None
        return
    parts = K.swiglu_gemm(gu.to(DEV), w.to(DEV))
    assert parts is not None and parts.dtype == torch.float32 and parts.shape[1:] == (M, N)
    assert parts.shape[0] == -(-I // 4096)
    act = P.plain_swiglu(gu.to(F64)[:, :I], gu.to(F64)[:, I:])
    _close(parts.sum(0), P.plain_linear(act, w.to(F64)), 6e-3)   # the activation is rounded to bfloat16 once


@pytest.mark.parametrize("M,I,Kd,bias", [(8, 16384, 4096, False), (3, 200, 96, True), (16, 331, 1032, False), (17, 331, 1032, True),
                                         (32, 4096, 4096, False), (5, 50, 8192, True), (24, 96, 200, False),
                                         (20, 8200, 1032, True), (2, 5760, 2304, False),
                                         # 33 to 64 rows, and 17 to 32 with a long K: chunks of X in LDS
                                         (64, 16384, 4096, False), (33, 331, 1032, True), (48, 200, 96, False), (49, 4100, 520, True),
                                         (40, 5760, 2304, False), (64, 61, 8, True), (20, 96, 8200, False)])
@pytest.mark.parametrize("tall", [False, True])
def test_gate_up_projection_with_the_activation_in_its_epilogue(K, monkeypatch, M, I, Kd, bias, tall):
    """One kernel for silu(x Wg^T) * (x Wu^T) against the plain formula and against the projection
    followed by the activation kernel (gate and up rounded to bfloat16 at the same place).  `tall`: from 17 rows
    the kernel with chunks of X in LDS where the outputs fill the chip; without it the kernel that keeps X in
    registers (up to 32 rows of a K up to 4096)."""
    monkeypatch.setattr(K, "USE_TALL", tall)
    if M > 32 or (M > 16 and Kd > 4096):   # rows that do not fit the registers
        if I < 12288 or not tall:
            # few outputs are left to the library on the engine's path (they do not fill the chip)
            assert K.gateup_swiglu_gemm(_rand((M, Kd), 31, torch.bfloat16).to(DEV), _rand((2 * I, Kd), 32, torch.bfloat16).to(DEV), None) is None
        if not tall:
            return
        monkeypatch.setattr(K, "GATEUP_TALL_MIN_OUTPUTS", 0)   # the kernel is tested all the same
    x, w = _rand((M, Kd), 31, torch.bfloat16), _rand((2 * I, Kd), 32, torch.bfloat16, scale=2.0 * Kd ** -0.5)
    b = _rand((2 * I,), 33, torch.bfloat16) if bias else None
    dev = lambda t: None if t is None else t.to(DEV)
    act = K.gateup_swiglu_gemm(dev(x), dev(w), dev(b))
    assert act is not None and act.shape == (M, I) and act.dtype == torch.bfloat16
    y = P.plain_linear(x.to(F64), w.to(F64), None if b is None else b.to(F64))
    _close(act, P.plain_swiglu(y[:, :I], y[:, I:]), 1e-2)
    two = K.swiglu(K.gemm(dev(x), dev(w), dev(b)))
    assert (act.float() - two.float()).abs().max() <= 2 ** -6 * max(float(two.float().abs().max()), 1e-6)
    assert K.gateup_swiglu_gemm(dev(x.float()), dev(w.float()), None) is None          # float32: not this kernel
    if M <= 32:
        big = _rand((209, Kd), 34, torch.bfloat16)
        assert K.gateup_swiglu_gemm(dev(big), dev(w), dev(b)) is None                  # too many rows


@pytest.mark.parametrize("M,N,K_", [(17, 200, 264), (64, 128, 1024), (65, 334, 520), (100, 4096, 4096), (128, 130, 16384),
                                    (129, 256, 640), (144, 4096, 16384), (208, 512, 2048), (97, 64, 72), (113, 1030, 4104),
                                    (32, 4096, 16384), (48, 2304, 5760)])
def test_products_with_chunks_of_x_in_lds(K, monkeypatch, M, N, K_):
    """`gemm_tall.hip`, both epilogues, chunks of 64 and of 128 k, weights in plain rows and in fragment order, against
    the plain formulas: K no multiple of a chunk, rows and outputs no multiple of a tile, one part and many."""
    from infinilm_amd.csrc import lib
    assert K.TALL_MAX_ROWS == lib.load().ilm_gemm_tall_max_rows()
    x, w = _rand((M, K_), 41, torch.bfloat16), _rand((N, K_), 42, torch.bfloat16, 0.05)
    want = P.plain_linear(x.to(F64), w.to(F64))
    kc, kb, cpp = K._tall_plan(M, N, K_)
    assert kc in (64, 128) and kb <= K.TALL_MAX_PARTS and kb == -(-(-(-K_ // kc)) // cpp)
    other = 192 - kc   # the other chunk length, split into three parts where there are that many chunks
    chunks = -(-K_ // other)
    cpp3 = -(-chunks // 3)
    for plan in ((kc, kb, cpp), (other, -(-chunks // cpp3), cpp3)):
        for fw in (None, K.pack_weight(w.to(DEV))):
            parts = K._gemm_tall(x.to(DEV), w.to(DEV), K_, fw, plan)
            assert parts.dtype == torch.float32 and parts.shape == (plan[1], M, N)
            _close(parts.sum(0), want, 1e-5)
    inter = N // 2
    bias = _rand((2 * inter,), 43, torch.bfloat16, 0.1)
    wg = w[:2 * inter]
    y = P.plain_linear(x.to(F64), wg.to(F64), bias.to(F64))
    want_act = P.plain_swiglu(y[:, :inter], y[:, inter:])
    two = K.swiglu(K.gemm(x.to(DEV), wg.to(DEV), bias.to(DEV)))
    for fw in (None, K.pack_weight(wg.to(DEV), "gate_up8")):
        for b, kc_ in ((bias.to(DEV), 128), (bias.to(DEV), 64), (None, 128)):
            act = K.gemm_tall_swiglu(x.to(DEV), wg.to(DEV), b, fw, kc_)
            assert act.shape == (M, inter) and act.dtype == torch.bfloat16
            if b is None:
                y0 = P.plain_linear(x.to(F64), wg.to(F64))
                _close(act, P.plain_swiglu(y0[:, :inter], y0[:, inter:]), 1e-2)
            else:
                _close(act, want_act, 1e-2)
                # gate and up are rounded to bfloat16 at the same place as the projection followed by the activation kernel
                assert (act.float() - two.float()).abs().max() <= 2 ** -6 * max(float(two.float().abs().max()), 1e-6)


def test_the_plan_of_a_product_with_parts():
    """Chunks of 128 k and a workgroup a compute unit; chunks of 64 and two a unit where a part would be longer than
    1024 k, up to 128 rows; never more than 16 parts."""
    from infinilm_amd import kernels as K
    assert K._tall_plan(64, 4096, 4096) == (128, 8, 4)       # o projection of the 8B shape: 32 tiles x 8 parts
    assert K._tall_plan(64, 4096, 16384) == (64, 16, 16)     # down projection: 32 tiles x 16 parts of 1024 k
    assert K._tall_plan(208, 4096, 16384) == (128, 8, 16)    # many rows: chunks of 128
    assert K._tall_plan(64, 2304, 5760) == (128, 15, 3)
    assert K._tall_plan(32, 128, 65536)[1] <= K.TALL_MAX_PARTS


def test_where_the_gate_up_projection_keeps_x_in_lds(K, monkeypatch):
    """17 to 112 rows, and up to 176 rows that are no multiple of 32, take the kernel with chunks of X in LDS
    when the outputs fill the chip; other row counts are left to the library's product and the activation kernel."""
    monkeypatch.setattr(K, "GATEUP_TALL_MIN_OUTPUTS", 0)
    w = _rand((2 * 96, 72), 44, torch.bfloat16, 0.1).to(DEV)
    for M, taken in ((17, True), (33, True), (65, True), (96, True), (112, True), (113, True), (128, False), (144, True), (160, False), (176, True), (192, False),
                     (175, True), (177, False), (208, False), (209, False)):
        x = _rand((M, 72), 45, torch.bfloat16).to(DEV)
        act = K.gateup_swiglu_gemm(x, w, None)
        assert (act is not None) == taken, M
        if taken:
            y = P.plain_linear(x.to(F64), w.to(F64))
            _close(act, P.plain_swiglu(y[:, :96], y[:, 96:]), 1e-2)


@pytest.mark.parametrize("M,Ko,H,I,bias,wdt", [(8, 4096, 4096, 16384, False, torch.bfloat16), (3, 96, 80, 200, True, torch.float32),
                                               (16, 1032, 328, 331, True, torch.bfloat16), (1, 2304, 2304, 5760, False, torch.float32),
                                               (20, 200, 96, 50, False, torch.float32), (32, 4096, 1024, 4096, True, torch.bfloat16),
                                               (5, 8192, 72, 61, False, torch.bfloat16)])
def test_branch_tail_and_deferred_norm(K, monkeypatch, M, Ko, H, I, bias, wdt):
    """The output projection with the residual sum and the first half of the next norm in its epilogue,
    and the gate/up projection that finishes that norm in its own: together they equal
    residual += alpha * (x Wo^T + b); swiglu(rmsnorm(residual) Wgu^T + b) of the plain formulas."""
    monkeypatch.setattr(K, "TAIL_MAX_ROWS", 32)
    x, wo = _rand((M, Ko), 51, torch.bfloat16), _rand((H, Ko), 52, torch.bfloat16, scale=2.0 * Ko ** -0.5)
    bo = _rand((H,), 53, torch.bfloat16) if bias else None
    r = _rand((M, H), 54, scale=2.0)
    nw = (_rand((H,), 55) * 0.2 + 1.0).to(wdt)
    wgu = _rand((2 * I, H), 56, torch.bfloat16, scale=2.0 * H ** -0.5)
    bgu = _rand((2 * I,), 57, torch.bfloat16) if bias else None
    dev = lambda t: None if t is None else t.to(DEV)
    alpha, eps = 0.37, 1e-5
    assert K.tail_ok(M, dev(wo), dev(bo), dev(nw), torch.bfloat16) and K.gateup_resident_ok(M, dev(wgu))
    rd = dev(r).clone()
    xw, ss = K.gemm_tail(dev(x), dev(wo), dev(bo), alpha, rd, dev(nw))
    act = K.gateup_swiglu_gemm(xw, dev(wgu), dev(bgu), row_ss=ss, eps=eps)
    r_want = r.to(F64) + P.plain_linear(x.to(F64), wo.to(F64), None if bo is None else bo.to(F64), alpha)
    _close(rd, r_want, 2e-5)
    assert rel_sum_sq(ss, rd, M) < 1e-5
    y = P.plain_linear(P.plain_rmsnorm(r_want, nw.to(F64), eps), wgu.to(F64), None if bgu is None else bgu.to(F64))
    _close(act, P.plain_swiglu(y[:, :I], y[:, I:]), 1.5e-2)
    # and against the three kernels it stands for (same places of rounding but one: r * w is rounded before the division)
    r2 = dev(r).clone()
    x2 = K.add_rmsnorm(r2, K.gemm(dev(x), dev(wo), dev(bo), 1.0, allow_parts=True), dev(nw), alpha, eps, torch.bfloat16)
    two = K.gateup_swiglu_gemm(x2, dev(wgu), dev(bgu))
    assert (act.float() - two.float()).abs().max() <= 2 ** -5 * max(float(two.float().abs().max()), 1e-6)
    _close(rd, r2, 1e-6)
    assert not K.tail_ok(33, dev(wo), dev(bo), dev(nw), torch.bfloat16)
    assert not K.tail_ok(M, dev(wo), dev(bo), dev(nw), torch.float32)


def rel_sum_sq(ss, r, M):
    """Relative error of the rows' sums of squares formed from the tiles' partial sums."""
    got = ss.to(F64).sum(0)[:M].cpu()
    want = (r.to(F64) ** 2).sum(1).cpu()
    return float(((got - want).abs() / want).max())


def _paged(k, v, page, n_pages, seed, dtype):
    """Scatters contiguous per-request keys/values [n, nkv, d] into a paged cache with a shuffled
    block table; unused slots hold large finite garbage so that a read beyond a length shows."""
    nkv, d = k[0].shape[1], k[0].shape[2]
    g = torch.Generator().manual_seed(seed)
    perm = torch.randperm(n_pages, generator=g).tolist()
    kc = torch.full((n_pages, nkv, page, d), 7.0, dtype=dtype)
    vc = torch.full((n_pages, nkv, d, page), -9.0, dtype=dtype)
    tables = []
    for kr, vr in zip(k, v):
        n = kr.shape[0]
        tab = [perm.pop() for _ in range(-(-n // page))]
        for i in range(n):
            kc[tab[i // page], :, i % page, :] = kr[i].to(dtype)
            vc[tab[i // page], :, :, i % page] = vr[i].to(dtype)
        tables.append(tab)
    width = max(len(t) for t in tables)
    bt = torch.full((len(tables), width), -1, dtype=torch.int32)
    for i, t in enumerate(tables):
        bt[i, :len(t)] = torch.tensor(t, dtype=torch.int32)
    return kc, vc, bt


def _attention_case(K, dtype, nh, nkv, d, page, lens, qlens, window=0, seed=0, spike=False, ramp=0.0):
    """Requests with `lens[i]` cached keys of which the last `qlens[i]` are this step's queries."""
    ks = [_rand((n, nkv, d), seed + 10 * i + 1, dtype) for i, n in enumerate(lens)]
    vs = [_rand((n, nkv, d), seed + 10 * i + 2, dtype) for i, n in enumerate(lens)]
    qs = [_rand((n, nh, d), seed + 10 * i + 3, dtype) for i, n in enumerate(lens)]
    if spike:
        # one far key per request must dominate: its score stands out by construction
        for q, k in zip(qs, ks):
            far = 3 if k.shape[0] > 3 else 0
            k[far] = (q[-1, 0:1, :].float() * 4.0 / math.sqrt(d)).to(dtype)
    if ramp:
        # scores of the last query's first head rise by `ramp` (natural units) a key: the running
        # maximum moves in every tile, by little or by much
        for q, k in zip(qs, ks):
            u = q[-1, 0, :].float()
            u = u / (u @ u)
            k[:, 0, :] = (k[:, 0, :].float() + torch.arange(k.shape[0])[:, None] * (ramp * math.sqrt(d)) * u).to(dtype)
    n_pages = sum(-(-n // page) for n in lens) + 3
    kc, vc, bt = _paged(ks, vs, page, n_pages, seed, dtype)
    q_rows, seg, pos = [], [], []
    for i, (n, ql) in enumerate(zip(lens, qlens)):
        q_rows.append(qs[i][n - ql:])
        seg += [i] * ql
        pos += list(range(n - ql, n))
    q = torch.cat(q_rows).reshape(-1, nh * d)
    # work lists as the step function builds them: runs of up to 8 tokens of a request, and single tokens
    tiles, singles, row = [], [], 0
    for ql in qlens:
        if ql == 1:
            singles.append(row)
        else:
            for k in range(0, ql, 8):
                tiles += [row + k, min(8, ql - k)]
        row += ql
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    extra = dict(tiles=i32(tiles).view(-1, 2), single_rows=i32(singles) if singles else None) if tiles else {}
    out = K.paged_attention(q.to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV), torch.tensor(seg, dtype=torch.int32, device=DEV),
                            torch.tensor(pos, dtype=torch.int32, device=DEV), nh, nkv, d, 1 / math.sqrt(d), window,
                            max_total_len=max(lens), **extra)
    want = []
    for i, (n, ql) in enumerate(zip(lens, qlens)):
        last = P.plain_attention(qs[i].to(F64), ks[i].to(F64), vs[i].to(F64), 1 / math.sqrt(d), window, first_row=n - ql)
        want.append(last.reshape(ql, nh * d))
    return out, torch.cat(want)


@pytest.mark.parametrize("nh,nkv,d,page", [(4, 2, 16, 4), (3, 1, 32, 8), (6, 3, 48, 16), (5, 5, 80, 7), (2, 1, 256, 16),
                                           (32, 2, 128, 64), (34, 2, 64, 12), (5, 1, 40, 8), (3, 3, 112, 20)])
def test_attention_float32(K, nh, nkv, d, page):
    """Heads in steps of 16 over pages that are multiples of 4 take the float matrix-core kernel (groups of up to
    16 heads side by side, groups of 17 in two parts); other head and page sizes the plain kernel."""
    out, want = _attention_case(K, torch.float32, nh, nkv, d, page, lens=[1, 70, 33, 130], qlens=[1, 70, 1, 5])
    _close(out, want, 3e-6)
    out, want = _attention_case(K, torch.float32, nh, nkv, d, page, lens=[90, 20], qlens=[2, 20], window=11, seed=5)
    _close(out, want, 3e-6)
    out, want = _attention_case(K, torch.float32, nh, nkv, d, page, lens=[300, 65], qlens=[1, 1], seed=9, spike=True)
    _close(out, want, 3e-6)


def test_attention_float32_one_wave_a_chunk_gives_the_same_bits(K, monkeypatch):
    """The plain kernel's two launch shapes (one wave walks all chunks of a token and head; one wave a
    chunk and a fold) agree bit for bit, so that a token decoded alone and the same token inside a
    portion of a prompt cannot differ."""
    case = dict(lens=[1500, 700, 513, 40], qlens=[1, 1, 3, 1])
    for window in (0, 600):
        monkeypatch.setattr(K, "BASIC_SPLIT", True)
        split, want = _attention_case(K, torch.float32, 6, 2, 48, 7, window=window, seed=4, **case)
        monkeypatch.setattr(K, "BASIC_SPLIT", False)
        whole, _ = _attention_case(K, torch.float32, 6, 2, 48, 7, window=window, seed=4, **case)
        assert torch.equal(split.cpu(), whole.cpu())
        _close(split, want, 3e-6)


@pytest.mark.parametrize("nh,nkv,d,page", [(6, 2, 48, 8), (32, 2, 128, 64), (17, 1, 32, 4)])
def test_attention_float32_matrix_cores_one_wave_a_chunk_gives_the_same_bits(K, monkeypatch, nh, nkv, d, page):
    """The float matrix-core kernel's two launch shapes agree bit for bit, with and without a window whose
    edge falls inside a chunk, and a token gives the same bits alone as inside a batch of portions."""
    case = dict(lens=[1500, 700, 513, 40], qlens=[1, 1, 3, 1])
    for window in (0, 600, 100):
        monkeypatch.setattr(K, "F32_ATTN_SPLIT", True)
        split, want = _attention_case(K, torch.float32, nh, nkv, d, page, window=window, seed=4, **case)
        monkeypatch.setattr(K, "F32_ATTN_SPLIT", False)
        whole, _ = _attention_case(K, torch.float32, nh, nkv, d, page, window=window, seed=4, **case)
        assert torch.equal(split.cpu(), whole.cpu())
        _close(split, want, 3e-6)
    monkeypatch.setattr(K, "F32_ATTN_SPLIT", True)
    alone, _ = _attention_case(K, torch.float32, nh, nkv, d, page, lens=[1500], qlens=[1], seed=4)
    among, _ = _attention_case(K, torch.float32, nh, nkv, d, page, lens=[1500, 700, 513], qlens=[40, 700, 2], seed=4)
    assert torch.equal(alone.cpu()[0], among.cpu()[39])


@pytest.mark.parametrize("nh,nkv,d", [(6, 2, 48), (3, 3, 64), (16, 1, 128), (2, 1, 256)])
@pytest.mark.parametrize("window", [0, 100, 21])
def test_attention_float32_pages_of_whole_tiles(K, monkeypatch, nh, nkv, d, window):
    """Pages that hold whole tiles of 16 keys are looked up once a tile, others once a lane: the same keys give the
    same bits either way, at the edges of tiles, chunks and windows and in both launch shapes."""
    case = dict(lens=[1, 16, 17, 128, 129, 300], qlens=[1, 1, 2, 1, 1, 3], window=window, seed=11)
    outs = []
    for split in (True, False):
        monkeypatch.setattr(K, "F32_ATTN_SPLIT", split)
        for page in (12, 16, 48):
            out, want = _attention_case(K, torch.float32, nh, nkv, d, page, **case)
            outs.append(out.cpu())
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    _close(outs[0], want, 3e-6)


@pytest.mark.parametrize("nh,nkv,d", [(4, 4, 64), (6, 1, 96), (4, 2, 128), (2, 2, 256)])
@pytest.mark.parametrize("window", [0, 20])
def test_attention_float32_short_contexts(K, monkeypatch, nh, nkv, d, window):
    """Contexts that end on either side of every second tile of a chunk, where a wave that walks all chunks may leave it early: the bits of
    a wave a chunk, and of pages looked up a lane at a time."""
    case = dict(lens=[1, 16, 31, 32, 33, 48, 63, 64, 65, 96, 128, 129, 160, 161, 192, 193], qlens=[1] * 16, window=window, seed=12)
    outs = []
    for split in (True, False):
        monkeypatch.setattr(K, "F32_ATTN_SPLIT", split)
        for page in (12, 16, 64):
            out, want = _attention_case(K, torch.float32, nh, nkv, d, page, **case)
            outs.append(out.cpu())
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    _close(outs[0], want, 3e-6)


@pytest.mark.parametrize("nh,nkv,d,page", [(32, 2, 128, 64), (17, 1, 64, 16), (10, 2, 64, 48), (12, 2, 128, 16), (4, 1, 128, 32), (3, 3, 64, 64),
                                           (4, 2, 128, 16)])
@pytest.mark.parametrize("window", [0, 100, 21])
def test_attention_float32_tiles_of_tokens_give_the_same_bits(K, monkeypatch, nh, nkv, d, page, window):
    """Portions whose tokens share their keys through LDS: every number of heads a wave and of tokens a tile, tiles that end on either side of a
    chunk, beside single tokens, against the kernel that takes tokens one by one."""
    case = dict(lens=[1, 2, 16, 17, 40, 128, 131, 300, 700, 523], qlens=[1, 2, 9, 17, 8, 3, 7, 300, 1, 12], window=window, seed=13)
    monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", 1 << 30)
    alone, want = _attention_case(K, torch.float32, nh, nkv, d, page, **case)
    monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", 0)
    for split in (True, False):
        monkeypatch.setattr(K, "F32_ATTN_SPLIT", split)
        tiles, _ = _attention_case(K, torch.float32, nh, nkv, d, page, **case)
        assert torch.equal(tiles.cpu(), alone.cpu())
    _close(tiles, want, 3e-6)


@pytest.mark.parametrize("nh,nkv,d", [(32, 2, 128), (10, 2, 64), (3, 3, 64)])
def test_attention_float32_cuts_tiles_and_single_rows_each_for_itself(K, monkeypatch, nh, nkv, d):
    """Either list in chunks with a fold of its own, both, neither, and in several launches that share a workspace: the bits of tokens one by one; what a list says of no token is skipped."""
    case = dict(lens=[1, 130, 300, 700, 523, 260], qlens=[1, 1, 21, 1, 12, 260], seed=14)
    monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", 1 << 30)
    alone, want = _attention_case(K, torch.float32, nh, nkv, d, 64, **case)
    monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", 0)
    rule, attention, pad = K.f32_attention, K.paged_attention, lambda t, row: torch.cat([row, t, row, row])
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    monkeypatch.setattr(K, "paged_attention", lambda *a, tiles, single_rows, **k: attention(*a, tiles=pad(tiles, i32([[0, 0]])),
                                                                                           single_rows=pad(single_rows, i32([-1])), **k))
    for tiles, rows, most in ((False, False, 8), (True, False, 1 << 20), (False, True, 1 << 20), (True, True, 1 << 20), (True, True, 8), (True, True, 24)):
        monkeypatch.setattr(K, "f32_attention", lambda *a: rule(*a)._replace(split_tiles=tiles, split_rows=rows, most=most, most_tiles=most // 8))
        out, _ = _attention_case(K, torch.float32, nh, nkv, d, 64, **case)
        assert torch.equal(out.cpu(), alone.cpu())
    # rows one by one without a list, in several launches
    monkeypatch.setattr(K, "paged_attention", attention)
    monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", 1 << 30)
    monkeypatch.setattr(K, "f32_attention", lambda *a: rule(*a)._replace(split_rows=True, most=100))
    out, _ = _attention_case(K, torch.float32, nh, nkv, d, 64, **case)
    assert torch.equal(out.cpu(), alone.cpu())
    _close(alone, want, 3e-6)


def test_attention_float32_lists_longer_than_a_launch_of_tiles(K, monkeypatch):
    """Tiles beyond a grid's second dimension, nearly all of them of no tokens, beside single rows: both cut into chunks, and the launches of tiles, which share
    the workspace, fold their own.  The bits of tokens one by one."""
    n, T = 200, 150
    k, v, q = (_rand((m, 1, 64), s, torch.float32) for m, s in ((n, 1), (n, 2), (T, 3)))
    kc, vc, bt = _paged([k], [v], 64, 6, 4, torch.float32)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    args = (q.reshape(T, 64).to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV), i32([0] * T), i32(list(range(n - T, n))), 1, 1, 64, 0.125)
    alone = K.paged_attention(*args, max_total_len=n)
    monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", 0)
    tiles = i32([[0, 0]] * 70000)
    tiles[:9], tiles[-9:] = i32([[8 * a, 8] for a in range(9)]), i32([[72 + 8 * a, 8] for a in range(9)])
    how = K.f32_attention(T, len(tiles), 6, 1, 1, 64, 64, n)
    assert how.tiled and how.split_tiles and how.split_rows and how.most_tiles < len(tiles) and 8 * len(tiles) + 6 <= how.most
    out = K.paged_attention(*args, max_total_len=n, tiles=tiles, single_rows=i32(list(range(144, T))))
    assert torch.equal(out.cpu(), alone.cpu())


@pytest.mark.parametrize("nh,nkv,d", [(32, 2, 128), (34, 2, 64), (10, 2, 64), (8, 2, 128), (3, 3, 64)])
@pytest.mark.parametrize("split", [False, True])
def test_attention_float32_gives_rows_of_no_request_zeros(K, monkeypatch, nh, nkv, d, split):
    """A recorded step's lists: tiles of no tokens, tiles of rows of no request, single rows of none.  Served rows have their bits, and nothing of what the
    results' and the workspace's memory held before is left in the others."""
    n, page, none = 300, 64, 19
    k, v, q = (_rand((m, h, d), s, torch.float32) for m, h, s in ((n, nkv, 1), (n, nkv, 2), (40 + 1 + none, nh, 3)))
    kc, vc, bt = _paged([k, k[:1]], [v, v[:1]], page, 8, 4, torch.float32)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    args = (q.reshape(-1, nh * d).to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV), i32([0] * 41 + [1] * none), i32(list(range(n - 40, n)) + [n - 1] + [0] * none), nh, nkv, d, 0.1)
    alone = K.paged_attention(*args, max_total_len=n)
    tiles = i32([[a, 8] for a in range(0, 40, 8)] + [[41, -8], [49, -8], [57, -3], [0, 0], [0, 0]])
    monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", 0)
    monkeypatch.setattr(K, "F32_ATTN_SPLIT", split)
    stale = [torch.full((m,), math.nan, device=DEV) for m in (alone.numel(), (8 * 10 + 4) * nh * 3 * (d + 4))]
    del stale
    out = K.paged_attention(*args, max_total_len=n, tiles=tiles, single_rows=i32([40, -1, -1, -1]))
    assert torch.equal(out[:41].cpu(), alone[:41].cpu()) and not out[41:].any()


@pytest.mark.parametrize("nh,nkv,d", [(9, 1, 64), (5, 1, 128), (3, 1, 64), (2, 2, 128)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attention_float32_tiles_keep_later_values_from_earlier_tokens(K, monkeypatch, nh, nkv, d, bad):
    """A value that is not finite reaches the tokens that see it and no other of the tile; what lies in the page behind the last token is not read."""
    n, first, page = 150, 101, 64
    k, v, q = (_rand((m, h, d), s, torch.float32) for m, h, s in ((n, nkv, 1), (n, nkv, 2), (n - first, nh, 3)))
    v[125, 0, 5] = bad
    kc, vc, bt = _paged([k], [v], page, 4, 4, torch.float32)
    for i in range(n, 192):
        kc[bt[0, i // page], :, i % page] = bad
        vc[bt[0, i // page], :, :, i % page] = bad
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    tiles = i32([[a, min(8, n - first - a)] for a in range(0, n - first, 8)])
    outs = []
    for most in (0, 1 << 30):
        monkeypatch.setattr(K, "F32_ATTN_TILE_MIN", most)
        outs.append(K.paged_attention(q.reshape(-1, nh * d).to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV), i32([0] * (n - first)), i32(list(range(first, n))),
                                      nh, nkv, d, 0.1, max_total_len=n, tiles=tiles).cpu())
    assert torch.isfinite(outs[0][:125 - first]).all() and not torch.isfinite(outs[0][125 - first:, 5]).any()
    assert torch.equal(torch.nan_to_num(outs[0], nan=7e30), torch.nan_to_num(outs[1], nan=7e30))


def test_attention_float32_refuses_a_bound_below_a_position_loudly(K):
    """A caller's bound on the lengths that is too small for a token must not lose a chunk silently: the
    fold marks the token's row with NaNs."""
    nh, nkv, d, page = 4, 2, 32, 16
    out, want = _attention_case(K, torch.float32, nh, nkv, d, page, lens=[700, 300], qlens=[1, 1], seed=2)
    _close(out, want, 3e-6)
    import infinilm_amd.kernels as kk
    orig = kk.paged_attention
    try:
        kk.paged_attention = lambda *a, **kw: orig(*a, **dict(kw, max_total_len=400))
        bad, _ = _attention_case(K, torch.float32, nh, nkv, d, page, lens=[700, 300], qlens=[1, 1], seed=2)
    finally:
        kk.paged_attention = orig
    assert torch.isnan(bad[0]).all() and not torch.isnan(bad[1]).any()


@pytest.mark.parametrize("nh,nkv,d,page", [(4, 2, 16, 16), (3, 1, 32, 16), (6, 3, 48, 32), (32, 2, 128, 64), (16, 16, 64, 16),
                                            (34, 2, 80, 16), (5, 1, 112, 48)])
def test_attention_bfloat16_matrix_cores(K, nh, nkv, d, page):
    # whole prompts, decode rows, a portion with history, lengths that cross key chunks of 256
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[1, 70, 33, 300], qlens=[1, 70, 1, 9])
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[700, 257, 256, 31], qlens=[1, 1, 1, 31], seed=3)
    _close(out, want, 1.2e-2)
    # a window's edge, inside a page and across chunks
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[90, 20, 600], qlens=[2, 20, 3], window=11, seed=5)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[600, 40], qlens=[1, 40], window=300, seed=6)
    _close(out, want, 1.2e-2)
    # a far key among hundreds must dominate
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[520, 65], qlens=[1, 1], seed=9, spike=True)
    _close(out, want, 1.2e-2)


@pytest.mark.parametrize("ramp", [0.02, 0.7, -0.05])
def test_attention_bfloat16_with_a_moving_maximum(K, ramp):
    """The tile kernel moves its exponent's reference point lazily: rising and falling scores."""
    out, want = _attention_case(K, torch.bfloat16, 32, 2, 128, 64, lens=[700, 130], qlens=[300, 130], seed=11, ramp=ramp)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, 6, 3, 48, 16, lens=[500, 9], qlens=[77, 9], seed=12, ramp=ramp, window=200)
    _close(out, want, 1.2e-2)


@pytest.mark.parametrize("d,page,window", [(128, 64, 128), (128, 64, 256), (64, 128, 192), (32, 256, 64)])
def test_attention_bfloat16_window_edge_on_a_tile_boundary(K, d, page, window):
    """A long portion under a window that is a multiple of the 64-key tile: one tile of tokens in
    eight has its last token's window begin exactly where a key tile begins, so that token sees
    nothing of the tile before (all its scores there are masked while it has seen no key yet) and
    the next tile takes the mask-free path."""
    out, want = _attention_case(K, torch.bfloat16, 4, 2, d, page, lens=[704, 333], qlens=[256, 200], window=window, seed=21)
    _close(out, want, 1.2e-2)


@pytest.mark.parametrize("nh,nkv,d,page", [(32, 2, 128, 256), (4, 2, 64, 128), (6, 3, 48, 256), (3, 1, 32, 128)])
def test_attention_bfloat16_pages_longer_than_a_key_tile(K, nh, nkv, d, page):
    """Pages of 128 and 256 keys: a 64-key tile begins in the middle of a page; portions with
    history, decoded tokens beside them, a far key that dominates."""
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[700, 300, 65, 1], qlens=[100, 1, 65, 1], seed=31)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[520, 900], qlens=[9, 1], seed=32, spike=True)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[600, 258], qlens=[77, 2], seed=33, window=130)
    _close(out, want, 1.2e-2)


@pytest.mark.parametrize("nh,nkv,d,page,lens", [(4, 2, 64, 64, [20000, 9000]), (8, 2, 128, 256, [16500]), (3, 1, 48, 16, [5000, 3300, 70])])
def test_attention_bfloat16_few_tokens_over_many_chunks(K, nh, nkv, d, page, lens):
    """One or two decoded tokens over tens of thousands of keys: up to 256 chunks, merged by the kernel of
    four waves (a quarter of the chunks each) instead of the one of one wave; a far key that dominates, a
    window that leaves most chunks out."""
    span, nsplit = K.attention_chunks(max(lens), page, K.bound_rows(len(lens)) * nkv, torch.device(DEV))
    assert nsplit > 24 and nsplit <= K.ATT_MAX_CHUNKS   # the merge of four waves
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=lens, qlens=[1] * len(lens), seed=41)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=lens, qlens=[1] * len(lens), seed=42, spike=True)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=lens, qlens=[1] * len(lens), seed=43, window=max(lens) // 2 + 77)
    _close(out, want, 1.2e-2)


@pytest.mark.parametrize("nh,nkv,d,page,n", [(8, 8, 64, 16, 40), (32, 2, 128, 64, 150), (4, 1, 32, 16, 120)])
def test_attention_bfloat16_many_single_tokens(K, nh, nkv, d, page, n):
    """Many decoded tokens in one launch: the chunks get long (several 128-key steps a workgroup,
    loads a step ahead), contexts from one key to a thousand."""
    g = torch.Generator().manual_seed(n)
    lens = torch.randint(1, 1000, (n,), generator=g).tolist()
    lens[0], lens[1], lens[2] = 1, 1000, 129
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=lens, qlens=[1] * n, seed=n)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=lens, qlens=[1] * n, seed=n + 1, window=200)
    _close(out, want, 1.2e-2)


@pytest.mark.parametrize("nh,nkv,d,page", [(16, 2, 64, 64), (32, 2, 128, 64), (3, 1, 48, 16), (20, 1, 112, 32), (4, 4, 16, 128)])
def test_attention_bfloat16_two_chunks_in_one_workgroup(K, monkeypatch, nh, nkv, d, page):
    """Up to 256 keys in chunks of 128: one workgroup merges the two chunks as the merge kernel does, bit for bit (that kernel
    serves when a third, empty chunk is asked for); contexts at the chunks' edges, a window that leaves the first out."""
    attention = K.paged_attention
    lens = [1, 31, 127, 128, 129, 160, 255, 256]
    for window, softcap, fw in ((0, 0.0, False), (100, 0.0, False), (0, 20.0, True)):
        got = []
        for chunks in (2, 3):
            monkeypatch.setattr(K, "attention_chunks", lambda *a: (K.ATT_STEP, chunks))
            monkeypatch.setattr(K, "paged_attention", lambda *a, **k: attention(*a, softcap=softcap, float_weights=fw, **k))
            out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=lens, qlens=[1] * len(lens), seed=60 + d, window=window)
            got.append(out.cpu())
        if not softcap:
            _close(got[0], want, 1.2e-2)
        assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("nh,nkv,d,page", [(1, 1, 64, 16), (4, 2, 128, 64), (8, 2, 16, 64), (3, 1, 96, 64), (5, 1, 128, 64), (12, 2, 64, 64), (16, 2, 48, 16), (8, 1, 128, 32),
                                           (9, 1, 64, 64)])
@pytest.mark.parametrize("window", [0, 64, 37])
def test_attention_bfloat16_tiles_of_few_heads(K, monkeypatch, nh, nkv, d, page, window):
    """Columns that hold one, two and four tokens: tiles that pair with the next one of their request and such that do not (a tile cut short, another
    request's, the last of an odd number), portions that end on either side of a key tile; with a softcap and float weights too."""
    attention = K.paged_attention
    case = dict(lens=[8, 9, 64, 65, 130, 40, 300, 17, 7, 200], qlens=[8, 9, 16, 63, 24, 5, 130, 1, 7, 33], seed=70 + d + nh, window=window)
    out, want = _attention_case(K, torch.bfloat16, nh, nkv, d, page, **case)
    _close(out, want, 1.2e-2)
    outs = []
    for tiles in (True, False):     # in tiles and one by one, under a softcap
        def both(*a, tiles=None, single_rows=None, _on=tiles, **k):
            return attention(*a, tiles=tiles if _on else None, single_rows=single_rows if _on else None, softcap=3.0, float_weights=True, **k)
        monkeypatch.setattr(K, "paged_attention", both)
        outs.append(_attention_case(K, torch.bfloat16, nh, nkv, d, page, **case)[0])
    _close(outs[0], outs[1], 1.2e-2)


def _tiles_of(K, nh, nkv, d, page, lists, positions, n, window=0, v=None, seg=None, seed=5):
    """bfloat16 attention of rows at `positions` of one request of `n` tokens, once for each list of tiles."""
    k, q = _rand((n, nkv, d), seed, BF16), _rand((len(positions), nh, d), seed + 1, BF16, 2.0)
    v = _rand((n, nkv, d), seed + 2, BF16) if v is None else v
    kc, vc, bt = _paged([k], [v], page, -(-n // page) + 2, 4, BF16)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    return [K.paged_attention(q.reshape(-1, nh * d).to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV), i32([0] * len(positions)), i32(positions), nh, nkv, d,
                              d ** -0.5, window, max_total_len=n, tiles=i32(x)).cpu() for x in lists]


@pytest.mark.parametrize("nh,nkv,d,page", [(32, 32, 64, 64), (64, 16, 128, 64), (48, 24, 96, 16), (48, 16, 128, 16)])
@pytest.mark.parametrize("first", [41, 56, 59, 63, 120])
@pytest.mark.parametrize("window", [0, 100])
def test_attention_bfloat16_pairs_of_tiles_give_the_bits_of_each(K, nh, nkv, d, page, first, window):
    """A token's result does not depend on whether its tile goes with the one beside it: where the two see different tiles of keys whole, too."""
    T = 44
    each = [[a, min(8, T - a)] for a in range(0, T, 8)]
    apart = [x for t in each for x in (t, [0, 0])]
    pairs, alone = _tiles_of(K, nh, nkv, d, page, (each, apart), list(range(first, first + T)), first + T, window)
    assert torch.equal(pairs, alone)


def test_attention_bfloat16_neighbouring_tiles_that_are_no_run(K):
    """Two tiles of the same request in neighbouring rows whose positions do not follow one another."""
    positions = list(range(0, 8)) + list(range(100, 108))
    both, first, second = _tiles_of(K, 2, 1, 64, 64, ([[0, 8], [8, 8]], [[0, 8]], [[8, 8]]), positions, 120)
    assert torch.equal(both, torch.cat([first[:8], second[8:]]))


def test_attention_bfloat16_with_a_block_table_beyond_lds(K):
    """33,000 keys in pages of 16: more block-table entries than the tile kernel keeps in LDS, and
    the most chunks the single-token kernel cuts a context into."""
    out, want = _attention_case(K, torch.bfloat16, 4, 2, 64, 16, lens=[33000, 50], qlens=[11, 1], seed=41)
    _close(out, want, 1.2e-2)
    out, want = _attention_case(K, torch.bfloat16, 4, 2, 64, 16, lens=[33000, 70], qlens=[1, 1], seed=42)
    _close(out, want, 1.2e-2)


def test_attention_does_not_depend_on_the_batch(K):
    """The same token alone and inside a larger batch gives the same bits (bfloat16 kernel), as long
    as both launches cut the context into chunks of the same length (few tokens: always 128 keys)."""
    nh, nkv, d, page = 8, 2, 64, 16
    out_a, _ = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[300], qlens=[1], seed=0)
    out_b, _ = _attention_case(K, torch.bfloat16, nh, nkv, d, page, lens=[300, 50, 700], qlens=[1, 50, 2], seed=0)
    assert torch.equal(out_a.cpu()[0], out_b.cpu()[0])


SAMPLE_ROWS = {   # name -> (row of logits, settings (temperature, top_k, top_p))
    "ties beyond the list": (lambda V, g: (torch.randn(V, generator=g) * 2).round(), [(1.0, 0, 0.7), (0.7, 3000, 1.0), (1.3, 50, 0.5)]),
    "all equal": (lambda V, g: torch.full((V,), 1.5), [(1.0, 0, 0.5), (1.0, 7, 0.9)]),
    "few values": (lambda V, g: torch.randint(0, 5, (V,), generator=g).float(), [(1.0, 0, 0.9), (0.5, 700, 0.95), (1.0, 3000, 0.999), (1.0, 0, 1.0)]),
    "half of them one value": (lambda V, g: torch.where(torch.rand(V, generator=g) < 0.5, 0.25, torch.randn(V, generator=g)), [(1.0, 0, 0.8), (1.0, 2500, 0.9)]),
    "close together": (lambda V, g: 0.5 + torch.randn(V, generator=g) * 0.01, [(1.0, 0, 0.9), (1.0, 50, 1.0), (5.0, 3000, 0.95), (0.02, 400, 1.0)]),
    "close together below a few": (lambda V, g: torch.where(torch.rand(V, generator=g) < 1e-4, 3.0, 0.5 + torch.randn(V, generator=g) * 1e-3),
                                   [(1.0, 0, 0.9), (1.0, 60, 1.0), (1.0, 3000, 0.5)]),
    "closer than a number's last bits": (lambda V, g: 1.0 + torch.randint(0, 5000, (V,), generator=g).float() * 2.0 ** -23, [(1.0, 0, 0.9), (1.0, 700, 1.0)]),
    "mostly masked": (lambda V, g: torch.where(torch.rand(V, generator=g) < 0.9, -math.inf, torch.randn(V, generator=g)), [(1.0, 0, 0.9), (0.8, 40, 0.9)]),
    "masked to the lowest number": (lambda V, g: torch.where(torch.rand(V, generator=g) < 0.999, -3.4028234663852886e38, torch.randn(V, generator=g)),
                                    [(1.0, 0, 0.9), (1.0, 5000, 1.0)]),
    "k in the last bin": (lambda V, g: torch.randn(V, generator=g) * 4, [(0.05, 60, 1.0), (0.05, 2500, 1.0), (0.02, 0, 0.999)]),
    "lists of any length": (lambda V, g: torch.randn(V, generator=g), [(1.0, 255, 0.9), (1.0, 256, 1.0), (1.0, 257, 0.95), (0.9, 1000, 0.95), (1.0, 1500, 1.0)]),
    "k beyond the list": (lambda V, g: torch.randn(V, generator=g), [(1.0, 2048, 1.0), (1.0, 2049, 0.95), (1.0, 6000, 0.9), (5.0, 0, 0.99)]),
}


@pytest.mark.parametrize("V", [1, 3, 255, 2049, 16385, 122753, 300001])
@pytest.mark.parametrize("name", list(SAMPLE_ROWS))
def test_sampling_where_thresholds_are_hard(K, name, V):
    """Every way to a threshold (list, radix, last bin) and to a token (list, tiles), rows that begin at any alignment, against the
    plain distribution.  A token's interval is met within 1e-6, less than a token has of the flattest rows: the plain masses are float64,
    the kernel's exponentials float32, good to four 2^-24 or so, as their running sums then are.  Masked entries are exact, and so
    are equal logits: of n that weigh the same u falls on number floor(u n)."""
    from infinilm_amd.csrc import lib
    make, settings = SAMPLE_ROWS[name]
    g = torch.Generator().manual_seed(V)
    row = make(V, g)
    row[0] = max(float(row[0]), 0.5)     # (one entry at least is not masked)
    us = [0.0, 1e-4, 0.13, 0.5, 0.77, 0.99, 1.0 - 2.0 ** -24]
    n = len(us)
    for temp, k, p in settings:
        mk = lambda v, dt: torch.tensor(v, dtype=dt, device=DEV)
        rows = row.expand(n, V).contiguous().to(DEV)
        rest = mk([temp] * n, torch.float32), mk([k] * n, torch.int32), mk([p] * n, torch.float32), mk(us, torch.float32)
        got = K.sample(rows, *rest).tolist()
        alone = torch.full((n,), -1, dtype=torch.int32, device=DEV)     # the same rows by one workgroup each, as many rows are
        assert lib.load().ilm_sample(alone.data_ptr(), rows.data_ptr(), *(t.data_ptr() for t in rest), None, n, V, V,
                                     torch.cuda.current_stream().cuda_stream) == 0
        assert alone.tolist() == got
        dist = P.plain_sample_distribution(row, temp, k, p)
        cdf = torch.cumsum(dist, 0)
        for u, tok in zip(us, got):
            assert 0 <= tok < V and dist[tok] > 0, f"token {tok} is outside the kept set (T={temp}, k={k}, p={p})"
            lo, hi = float(cdf[tok] - dist[tok]), float(cdf[tok])
            assert lo - 1e-6 <= u <= hi + 1e-6, f"u={u} not in token {tok}'s interval [{lo}, {hi}] (T={temp}, k={k}, p={p})"
            assert name != "all equal" or tok == int(torch.tensor(u, dtype=torch.float32).item() * V)


@pytest.mark.parametrize("n,V", [(32, 40961), (33, 98304), (33, 98305), (64, 98305), (64, 122753), (65, 122753)])
def test_sampling_many_long_rows(K, n, V):
    """Either side of where rows are cut into chunks, every row with settings of its own: the tokens of one workgroup a row."""
    from infinilm_amd.csrc import lib
    g = torch.Generator(device=DEV).manual_seed(n + V)
    rows = torch.randn((n, V), generator=g, device=DEV) * 2
    rows[::5] = rows[::5].round()
    i = torch.arange(n, device=DEV)
    rest = (0.5 + 0.1 * (i % 7).float(), ((i * 37) % 11 * (i % 3) * 40).to(torch.int32), 1.0 - 0.06 * (i % 4).float(),
            torch.rand(n, generator=g, device=DEV))
    alone = torch.full((n,), -1, dtype=torch.int32, device=DEV)
    assert lib.load().ilm_sample(alone.data_ptr(), rows.data_ptr(), *(t.data_ptr() for t in rest), None, n, V, V,
                                 torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(K.sample(rows, *rest), alone)


@pytest.mark.parametrize("V", [300, 30000, 50000])
def test_sampling_rows_with_nan_and_infinity(K, V):
    """Whatever a row holds, the token is one of its own; a NaN is drawn only where nothing else is kept."""
    g = torch.Generator().manual_seed(V)
    rows = torch.randn((6, V), generator=g) * 2
    rows[0, ::7] = math.nan
    rows[1, 5] = math.inf
    rows[2, 9::3] = math.inf
    rows[3] = -math.inf
    rows[4] = math.nan
    rows[5, V - 1] = math.nan
    mk = lambda v, dt: torch.tensor([v] * 6, dtype=dt, device=DEV)
    for temp, k, p in ((1.0, 0, 0.9), (0.7, 0, 1.0), (1.0, 40, 0.9), (1.0, V - 1, 1.0)):
        got = K.sample(rows.to(DEV), mk(temp, torch.float32), mk(k, torch.int32), mk(p, torch.float32), mk(0.4, torch.float32)).tolist()
        assert all(0 <= t < V for t in got)
        assert not math.isnan(float(rows[5, got[5]])) and not math.isnan(float(rows[0, got[0]]))


@pytest.mark.parametrize("V", [300, 5000, 50000])
def test_sampling_under_a_negative_temperature(K, V):
    """No request can have one, but a caller of the kernel can: it turns the kept tokens' order of probabilities around and stays inside its
    histogram."""
    g = torch.Generator().manual_seed(V)
    row = torch.rand(V, generator=g)
    us = [0.0, 0.3, 0.9, 1.0 - 2.0 ** -24]
    for temp, k in ((-0.5, 0), (-2.0, 40), (-1.0, 3000)):
        mk = lambda v, dt: torch.tensor(v, dtype=dt, device=DEV)
        got = K.sample(row.expand(4, V).contiguous().to(DEV), mk([temp] * 4, torch.float32), mk([k] * 4, torch.int32), mk([1.0] * 4, torch.float32),
                       mk(us, torch.float32)).tolist()
        keep = row >= torch.sort(row, descending=True).values[k - 1] if 0 < k < V else torch.ones(V, dtype=torch.bool)
        cdf = torch.cumsum(torch.where(keep, torch.exp(row.to(F64) / temp), torch.zeros(V, dtype=F64)), 0)
        cdf /= cdf[-1].clone()
        for u, tok in zip(us, got):
            assert 0 <= tok < V and keep[tok] and (float(cdf[tok - 1]) if tok else 0.0) - 1e-6 <= u <= float(cdf[tok]) + 1e-6


def test_argmax_and_sampling(K):
    V = 73448
    logits = _rand((5, V), 20, scale=3.0)
    logits[1, 100] = logits[1, 70000] = 50.0      # a tie: the first index wins
    logits[2, V - 1] = 60.0
    dl = logits.to(DEV)
    assert K.argmax(dl).tolist() == [int(torch.argmax(logits[0])), 100, V - 1, int(torch.argmax(logits[3])), int(torch.argmax(logits[4]))]

    def run(temp, k, p, u, rows=logits):
        n = rows.shape[0]
        mk = lambda v, dt: torch.tensor([v] * n if not isinstance(v, list) else v, dtype=dt, device=DEV)
        return K.sample(rows.to(DEV), mk(temp, torch.float32), mk(k, torch.int32), mk(p, torch.float32),
                        mk(u, torch.float32)).tolist()

    assert run(1.0, 1, 1.0, 0.5) == K.argmax(dl).tolist()           # top_k 1 is greedy
    # a greedy row beside sampled rows, index 0 tied for the maximum: the first index wins there too
    tie = logits.clone()
    tie[0, 0] = tie[0, 5000] = tie[3, 0] = tie[3, V - 1] = 70.0
    mixed = run([0.0, 1.0, 0.8, 1.0, 0.0], [0, 1, 40, 1, 0], 1.0, 0.3, tie)
    assert mixed[0] == 0 and mixed[3] == 0 and mixed[1] == 100 and mixed[4] == int(torch.argmax(logits[4]))
    assert run(0.0, 0, 1.0, 0.9) == K.argmax(dl).tolist()           # temperature 0 is greedy
    # inverse CDF in vocabulary order against the plain implementation, over many u
    small = _rand((1, 331), 21, scale=2.0)
    for temp, k, p in [(0.8, 0, 1.0), (1.3, 5, 1.0), (1.0, 0, 0.6), (0.7, 40, 0.9), (1.0, 331, 1.0), (2.0, 2, 0.5)]:
        dist = P.plain_sample_distribution(small[0], temp, k, p)
        cdf = torch.cumsum(dist, 0)
        us = [i / 64.0 + 1 / 128.0 for i in range(64)]
        got = run(temp, k, p, us, small.expand(64, 331).contiguous())
        for u, tok in zip(us, got):
            assert dist[tok] > 0, f"token {tok} is outside the kept set (T={temp}, k={k}, p={p})"
            lo = float(cdf[tok] - dist[tok])
            assert lo - 1e-4 <= u <= float(cdf[tok]) + 1e-4, f"u={u} not in token {tok}'s interval"
    # every row length takes its own kernel shape (row in registers of 1024 or 512 threads, or streamed)
    for Vn in (16384, 20000, 40000, 73448, 90000, 122753):
        big = _rand((1, Vn), 30 + Vn % 7, scale=2.5)
        for temp, k, p in [(0.9, 0, 1.0), (1.1, 50, 0.9), (1.0, 0, 0.7), (0.6, 7, 1.0)]:
            dist = P.plain_sample_distribution(big[0], temp, k, p)
            cdf = torch.cumsum(dist, 0)
            us = [i / 8.0 + 1 / 16.0 for i in range(8)]
            got = run(temp, k, p, us, big.expand(8, Vn).contiguous())
            for u, tok in zip(us, got):
                assert dist[tok] > 0, f"V={Vn}: token {tok} is outside the kept set (T={temp}, k={k}, p={p})"
                lo = float(cdf[tok] - dist[tok])
                assert lo - 2e-4 <= u <= float(cdf[tok]) + 2e-4, f"V={Vn}: u={u} not in token {tok}'s interval"
    # frequencies over many draws follow the probabilities
    dist = P.plain_sample_distribution(small[0], 1.0, 8, 1.0)
    n = 4096
    g = torch.Generator().manual_seed(1)
    us = torch.rand(n, generator=g).tolist()
    got = torch.tensor(run(1.0, 8, 1.0, us, small.expand(n, 331).contiguous()))
    freq = torch.bincount(got, minlength=331).to(F64) / n
    assert float((freq - dist).abs().max()) < 0.03
    # the big vocabulary: top-k keeps exactly the k largest
    top = set(torch.topk(logits[0], 3).indices.tolist())
    for u in (0.01, 0.4, 0.99):
        assert run(1.5, 3, 1.0, u, logits[:1])[0] in top


@pytest.mark.parametrize("V", [4095, 4096, 4099, 40003, 122753])
@pytest.mark.parametrize("name", ["normal", "few values", "mostly masked", "close together", "sorted", "NaN", "infinity"])
def test_sampling_top_k_of_few(K, name, V):
    """A top-k that one reading of a row may give, at the ends of its range and of the lists it takes, beside rows that it leaves to the
    histograms: the plain distribution's intervals (within 1e-6, see test_sampling_where_thresholds_are_hard), and where NaN and infinities leave
    none, the tokens that rows in chunks give."""
    g = torch.Generator().manual_seed(V + 1)
    row = {"normal": lambda: torch.randn(V, generator=g) * 2,
           "few values": lambda: torch.randint(0, 40, (V,), generator=g).float(),
           "mostly masked": lambda: torch.where(torch.rand(V, generator=g) < 0.99, -math.inf, torch.randn(V, generator=g)),
           "close together": lambda: 3.0 + torch.randn(V, generator=g) * 1e-4,
           "sorted": lambda: torch.randn(V, generator=g).sort().values,
           "NaN": lambda: torch.where(torch.rand(V, generator=g) < 0.1, math.nan, torch.randn(V, generator=g)),
           "infinity": lambda: torch.randn(V, generator=g)}[name]()
    if name == "infinity":
        row[V // 3], row[V // 2] = math.inf, -math.inf
    most = K.sample_few_k()
    us = [0.0, 0.3, 0.71, 1.0 - 2.0 ** -24]
    n = len(us)
    mk = lambda v, dt: torch.tensor(v, dtype=dt, device=DEV)
    rows = row.expand(n, V).contiguous().to(DEV)
    for k in (2, 3, 50, 63, 64, 65, 128, most, most + 1):
        for p in (1.0, 0.9, 1e-3):
            prm = torch.cat([mk([0.8] * n, torch.float32), mk([k] * n, torch.int32).view(torch.float32), mk([p] * n, torch.float32), mk(us, torch.float32)])
            one, cut = K.sample_packed(rows, prm, few=True).tolist(), K.sample_packed(rows, prm).tolist()
            assert one == cut
            if name in ("NaN", "infinity"):
                assert all(row[t] == row[t] for t in one)
                continue
            dist = P.plain_sample_distribution(row, 0.8, k, p)
            cdf = torch.cumsum(dist, 0)
            for u, tok in zip(us, one):
                assert 0 <= tok < V and dist[tok] > 0, f"token {tok} is outside the kept set (k={k}, p={p})"
                assert float(cdf[tok] - dist[tok]) - 1e-6 <= u <= float(cdf[tok]) + 1e-6


BF16 = torch.bfloat16
PORTION_SIZES = [(33, 8, 64), (64, 200, 128), (65, 1000, 192), (127, 129, 256), (128, 64, 320), (129, 257, 448), (300, 520, 1024), (513, 1032, 576)]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K_", PORTION_SIZES)
def test_portion_product(K, M, N, K_, bias):
    """Every tile at edges of rows, outputs and stages (fewer stages than the kernel holds, just as many, more), into rows of any stride.
    An output is a float sum (off by at most K 2^-24 of the sum of its terms' sizes) rounded to bfloat16 (2^-8 of it)."""
    g = torch.Generator().manual_seed(M * 31 + N)
    x, w = (torch.randn(s, generator=g).to(BF16).to(DEV) for s in ((M, K_ + 8), (N, K_ + 16)))
    x, w = x[:, 8:], w[:, :K_]
    b = torch.randn(N, generator=g).to(BF16).to(DEV) if bias else None
    want = x.double() @ w.double().T + (b.double() if bias else 0.0)
    size = x.double().abs() @ w.double().abs().T + (b.double().abs() if bias else 0.0)
    first = None
    for tile in (1, 2, 3):
        for pad in (0, 3, 8):
            c = torch.full((M, N + pad), 7.0, dtype=BF16, device=DEV)
            K.portion_gemm(x, w, b, c[:, :N], tile)
            assert torch.equal(c[:, N:], torch.full_like(c[:, N:], 7.0))
            err = (c[:, :N].double() - want).abs()
            assert bool((err <= want.abs() * 2.0 ** -8 + size * K_ * 2.0 ** -23).all()), (tile, pad)
            first = c[:, :N].clone() if first is None else first
            assert torch.equal(c[:, :N], first), (tile, pad)     # one order of sums, whatever the tile


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,N,K_", PORTION_SIZES)
def test_portion_gate_and_up(K, M, N, K_, act):
    """The same sums as the product's, and the activation kernel's results on them."""
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K_), generator=g).to(BF16).to(DEV), (torch.randn((2 * N, K_), generator=g) / math.sqrt(K_)).to(BF16).to(DEV)
    for b in (None, torch.randn(2 * N, generator=g).to(BF16).to(DEV)):
        want = K.swiglu(K.portion_gemm(x, w, b, torch.empty((M, 2 * N), dtype=BF16, device=DEV), 1), act)
        for tile in (1, 4, 5):
            assert torch.equal(K.portion_glu(x, w, b, act, tile), want), tile


@pytest.mark.parametrize("nh,nkv,d", [(3, 1, 32), (4, 2, 64), (5, 5, 96), (8, 2, 128)])
@pytest.mark.parametrize("M", [65, 130, 333])
def test_portion_qkv(K, M, nh, nkv, d):
    """The product's sums, and what the rotation's kernel makes of them, in the queries' rows and in the cache; tokens without a slot
    write nothing.  The two kernels may round a rotated value differently by its last bit (a sum of two products, contracted or not)."""
    g = torch.Generator().manual_seed(M + d)
    K_, page, pages = 192, 16, M // 16 + 2
    N = (nh + 2 * nkv) * d
    x, w = torch.randn((M, K_), generator=g).to(BF16).to(DEV), (torch.randn((N, K_), generator=g) / math.sqrt(K_)).to(BF16).to(DEV)
    cos, sin = (torch.randn((500, d // 2), generator=g).to(DEV) for _ in range(2))
    pos = torch.randint(0, 500, (M,), generator=g, dtype=torch.int32).to(DEV)
    slots = torch.randperm(page * pages, generator=g)[:M].to(torch.int32)
    slots[::7] = -1
    slots = slots.to(DEV)
    for b in (None, torch.randn(N, generator=g).to(BF16).to(DEV)):
        rows = K.portion_gemm(x, w, b, torch.empty((M, N), dtype=BF16, device=DEV), 1)
        kc, vc = torch.zeros((pages, nkv, page, d), dtype=BF16, device=DEV), torch.zeros((pages, nkv, d, page), dtype=BF16, device=DEV)
        K.rope_kvwrite(rows, pos, cos, sin, kc, vc, slots, nh, nkv, d, d)
        for tile in (1, 2):
            for s in (slots, None):
                kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
                q = K._qkv_rope(x, w, b, pos, cos, sin, kc2, vc2, s, nh, nkv, d, tile)
                near = lambda a, c: bool(((a.double() - c.double()).abs() <= c.double().abs() * 2.0 ** -7 + 1e-6).all())
                assert near(q, rows[:, :nh * d])
                if s is None:
                    assert not kc2.any() and not vc2.any()
                else:
                    assert near(kc2, kc) and torch.equal(vc2, vc)


def test_portion_rule(K):
    """The rule takes what the kernels take: K in steps of 64, one round of tiles, and the public entry points go there and give
    the library path's results to rounding."""
    dev = torch.device(DEV)
    assert K._portion_tile("plain", 2048, 1024, 1000, dev) == 0 and K._portion_tile("glu", 300, 8192, 2048, dev) == 0
    for M, N, K_ in ((2048, 1024, 1024), (300, 1024, 1024), (65, 8192, 1024), (600, 4096, 2048)):
        tile = K._portion_tile("plain", M, N, K_, dev)
        assert tile in (1, 2, 3)
        g = torch.Generator(device=DEV).manual_seed(M)
        x, w = torch.randn((M, K_), generator=g, device=DEV).to(BF16), torch.randn((N, K_), generator=g, device=DEV).to(BF16)
        want = x.float() @ w.float().T
        got = K.gemm(x, w)
        assert torch.equal(got, K.portion_gemm(x, w, None, torch.empty_like(got), tile))
        assert float((got.float() - want).norm() / want.norm()) < 2.0 ** -8
    # gate/up and q/k/v: the forms that end in what their next kernel did, against the product and that kernel (see test_portion_qkv on the rotation)
    g = torch.Generator(device=DEV).manual_seed(2)
    for M in (300, 700):
        x, w = torch.randn((M, 1024), generator=g, device=DEV).to(BF16), (torch.randn((8192, 1024), generator=g, device=DEV) / 32).to(BF16)
        assert K._portion_tile("glu", M, 8192, 1024, dev)
        y = K.gateup_swiglu_gemm(x, w, None)
        assert y is not None and torch.equal(y, K.swiglu(K.portion_gemm(x, w, None, torch.empty((M, 8192), dtype=BF16, device=DEV), 1), "silu"))
    for M in (300, 1000, 2048):
        x, w = torch.randn((M, 1024), generator=g, device=DEV).to(BF16), (torch.randn((1280, 1024), generator=g, device=DEV) / 32).to(BF16)
        pos, slots = torch.arange(M, dtype=torch.int32, device=DEV), torch.arange(M, dtype=torch.int32, device=DEV)
        cos, sin = torch.rand((M, 32), generator=g, device=DEV), torch.rand((M, 32), generator=g, device=DEV)
        caches = [(torch.zeros((M // 16 + 1, 2, 16, 64), dtype=BF16, device=DEV), torch.zeros((M // 16 + 1, 2, 64, 16), dtype=BF16, device=DEV)) for _ in range(2)]
        assert K._portion_tile("rope", M, 1280, 1024, dev)
        q = K.qkv_rope_gemm(x, w, None, pos, cos, sin, *caches[0], slots, 16, 2, 64, 64)
        rows = K.portion_gemm(x, w, None, torch.empty((M, 1280), dtype=BF16, device=DEV), 1)
        K.rope_kvwrite(rows, pos, cos, sin, *caches[1], slots, 16, 2, 64, 64)
        assert q is not None and torch.equal(caches[0][1], caches[1][1])
        for got, want in ((q, rows[:, :1024]), (caches[0][0], caches[1][0])):
            assert bool(((got.double() - want.double()).abs() <= want.double().abs() * 2.0 ** -7 + 1e-6).all())


@pytest.mark.parametrize("M,K_,nh,nkv,d,parts", [(1, 256, 2, 1, 32, 1), (1, 1024, 16, 2, 64, 4), (2, 1024, 5, 1, 64, 8), (1, 2048, 16, 2, 64, 2), (8, 256, 3, 3, 96, 3),
                                                 (1, 3328, 4, 4, 64, 3), (1, 4096, 32, 2, 128, 4), (2, 768, 6, 2, 128, 5)])
def test_qkv_projection_that_forms_its_rows(K, M, K_, nh, nkv, d, parts):
    """Against the norm's kernel and the projection one after the other.  The new residual rows are the same sums; the norm's sum of squares
    is taken in another order (some 2^-22 of it), which can turn a normed value's last bit (2^-8), and by that an output by at
    most 2^-8 of a thousandth or so of its terms: held to 2^-6 of the largest output of a row."""
    g = torch.Generator().manual_seed(M * K_ + d)
    page, pages, N = 16, 4, (nh + 2 * nkv) * d
    r, h = torch.randn((M, K_), generator=g).to(DEV) * 3, torch.randn((parts, M, K_), generator=g).to(DEV)
    w = (torch.randn((N, K_), generator=g) / math.sqrt(K_)).to(BF16).to(DEV)
    nw = (1 + 0.1 * torch.randn(K_, generator=g)).to(DEV)
    b = torch.randn(N, generator=g).to(BF16).to(DEV)
    cos, sin = (torch.randn((64, d // 2), generator=g).to(DEV) for _ in range(2))
    pos = torch.randint(0, 64, (M,), generator=g, dtype=torch.int32).to(DEV)
    slots = torch.randperm(page * pages, generator=g)[:M].to(torch.int32).to(DEV)
    if M > 2:
        slots[1] = -1
    for nw_, off, bias in ((nw, 0.0, None), (nw.to(BF16), 1.0, b)):
        c1, c2 = ([torch.zeros((pages, nkv, page, d), dtype=BF16, device=DEV), torch.zeros((pages, nkv, d, page), dtype=BF16, device=DEV)] for _ in range(2))
        before = r.clone()
        q, new = K.qkv_rope_sum(r, h, 0.7, nw_, off, 1e-5, w, bias, pos, cos, sin, *c1, slots, nh, nkv, d, d)
        assert torch.equal(r, before)
        want = r.clone()
        x = K.add_rmsnorm(want, h, nw_, 0.7, 1e-5, BF16, weight_offset=off)
        assert float((new - want).abs().max()) <= 2.0 ** -22 * float(want.abs().max() + h.abs().sum(0).max())
        ref = K.qkv_rope_gemm(x, w, bias, pos, cos, sin, *c2, slots, nh, nkv, d, d)
        for got, exp in ((q, ref), (c1[0], c2[0]), (c1[1], c2[1])):
            assert float((got.float() - exp.float()).abs().max()) <= 2.0 ** -6 * float(exp.float().abs().max())
            assert torch.equal(got == 0, exp == 0) or float(((got == 0) != (exp == 0)).float().mean()) < 1e-3
    more = torch.zeros((parts, 9, K_), device=DEV)      # (more rows than a workgroup forms)
    assert K.qkv_rope_sum(more[0], more, 1.0, nw, 0.0, 1e-5, w, None, pos, cos, sin, None, None, None, nh, nkv, d, d) is None
    assert K.qkv_rope_sum(r[:, :K_ - 8].contiguous(), h[:, :, :K_ - 8].contiguous(), 1.0, nw[:K_ - 8], 0.0, 1e-5, w[:, :K_ - 8].contiguous(), None, pos, cos, sin,
                          None, None, None, nh, nkv, d, d) is None


@pytest.mark.parametrize("M,N,K_,parts", [(8, 1024, 8192, 8), (16, 2304, 5760, 6), (1, 4099, 4104, 5), (3, 1030, 8200, 3), (2, 1023, 8192, 2)])
def test_gemm_few_rows_in_short_parts_of_a_long_k(K, M, N, K_, parts):
    """Either side of where K beyond 4,096 is cut into parts of 1,024: the parts' float sum against float64, as in
    test_gemm_few_rows_in_short_parts, and the norm that sums them."""
    a, w = _rand((M, K_), 60, torch.bfloat16), _rand((N, K_), 61, torch.bfloat16)
    got = K.gemm(a.to(DEV), w.to(DEV), allow_parts=True)
    assert got.dtype == torch.float32 and got.shape == (parts, M, N)
    want = P.plain_linear(a.to(F64), w.to(F64))
    _close(got.sum(0), want, 2e-6 * math.sqrt(K_))
    r = torch.zeros((M, N), dtype=torch.float32, device=DEV)
    K.add_rmsnorm(r, got, torch.ones(N, dtype=torch.bfloat16, device=DEV), 1.0, 1e-6, torch.bfloat16)
    _close(r, want, 2e-6 * math.sqrt(K_))


def test_a_top_k_that_is_no_int(K):
    """Rows whose top-k is a float, or beyond 32 bits, beside others: the tokens of the whole number, and of the whole vocabulary."""
    from infinilm_amd import SamplingParams
    from infinilm_amd.sampling import Sampler
    logits = torch.randn((3, 5000), generator=torch.Generator().manual_seed(3)).to(DEV)
    rows = lambda ks: [(SamplingParams(top_k=k, top_p=0.9), i, 4) for i, k in enumerate(ks)]
    want = Sampler(5).sample(logits, rows([50, 4, 0]))
    assert Sampler(5).sample(logits, rows([50.0, 4.5, 2 ** 31])) == want


@pytest.mark.parametrize("V", [4096, 40003, 122753])
@pytest.mark.parametrize("name", ["masked to 60", "masked to 3", "finite mask", "all equal", "two values", "zeros of both signs", "cold", "ties and a mask", "steps", "NaN and a mask"])
def test_sampling_top_k_of_few_that_ends_in_ties_or_in_a_mask(K, name, V):
    """The bound of a top-k of few where nothing above it reaches k: elements that no number can draw below, or ties, whose whole number is kept.
    The plain distribution's intervals (within 1e-6, see test_sampling_where_thresholds_are_hard), and the tokens that rows in chunks give."""
    g = torch.Generator().manual_seed(V + 2)
    row = torch.randn(V, generator=g) * 2
    some = torch.randperm(V, generator=g)
    temp = 0.02 if name == "cold" else 0.8
    if name == "masked to 60":
        row[some[60:]] = -math.inf
    elif name == "masked to 3":
        row[some[3:]] = -math.inf
    elif name == "finite mask":
        row[some[60:]] = -3e38
    elif name == "all equal":
        row[:] = 1.25
    elif name == "two values":
        row[:] = -1.0
        row[some[:30]] = 0.5
    elif name == "zeros of both signs":
        row = -row.abs() - 1
        row[some[:500]] = 0.0
        row[some[500:1000]] = -0.0
    elif name == "ties and a mask":
        row[some[2000:]] = -math.inf
        row[some[:2000]] = torch.randint(0, 3, (2000,), generator=g).float()
    elif name == "steps":
        row = (row * 2).round() / 2
    elif name == "NaN and a mask":
        row[some[100:]] = -math.inf
        row[some[:40]] = math.nan
    us = [0.0, 0.3, 0.71, 1.0 - 2.0 ** -24]
    mk = lambda v, dt: torch.tensor(v, dtype=dt, device=DEV)
    rows = row.expand(4, V).contiguous().to(DEV)
    for k in (2, 50, 100, 191, 192, K.sample_few_k()):
        for p in (1.0, 0.9, 1e-3):
            prm = torch.cat([mk([temp] * 4, torch.float32), mk([k] * 4, torch.int32).view(torch.float32), mk([p] * 4, torch.float32), mk(us, torch.float32)])
            one = K.sample_packed(rows, prm, few=True).tolist()
            assert one == K.sample_packed(rows, prm).tolist()
            if name == "NaN and a mask":
                assert all(row[t] == row[t] and row[t] > -math.inf for t in one)
                continue
            if name == "zeros of both signs":      # (their keys differ, so where a top-k ends among them it ends at the sign)
                if k > 500:
                    continue
                dist = P.plain_sample_distribution(torch.where((row == 0) & (torch.signbit(row)), -1.0, row), temp, k, p)
            else:
                dist = P.plain_sample_distribution(row, temp, k, p)
            cdf = torch.cumsum(dist, 0)
            for u, tok in zip(us, one):
                assert 0 <= tok < V and dist[tok] > 0, f"token {tok} is outside the kept set (k={k}, p={p})"
                assert float(cdf[tok] - dist[tok]) - 1e-6 <= u <= float(cdf[tok]) + 1e-6


@pytest.mark.parametrize("shared", ["x", "w"])
def test_products_of_rows_that_share_memory(K, shared):
    """One row for all (an expanded tensor), at sizes whose portions have a kernel of their own: the product, gate/up with its activation and
    q/k/v with rotation give what the rows one by one give, or leave the call to who takes it.  (Tolerance: bfloat16 results.)"""
    g = torch.Generator().manual_seed(9)
    M, N, k = 300, 1024, 1024
    x, w = torch.randn((M, k), generator=g).to(BF16).to(DEV), (torch.randn((N, k), generator=g) / 32).to(BF16).to(DEV)
    x, w = (x[:1].expand(M, k), w) if shared == "x" else (x, w[:1].expand(N, k))
    want = x.float() @ w.float().T
    assert float((K.gemm(x, w).float() - want).abs().max()) <= 2.0 ** -7 * float(want.abs().max())
    y = K.gateup_swiglu_gemm(x, w, None)
    if y is not None:
        want_y = torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:]
        assert float((y.float() - want_y).abs().max()) <= 2.0 ** -6 * float(want_y.abs().max())
    pos = torch.zeros(M, dtype=torch.int32, device=DEV)
    cos, sin = torch.ones((4, 32), device=DEV), torch.zeros((4, 32), device=DEV)
    q = K.qkv_rope_gemm(x, w, None, pos, cos, sin, None, None, None, 12, 2, 64, 64)
    if q is not None:
        assert float((q.float() - want[:, :768]).abs().max()) <= 2.0 ** -7 * float(want.abs().max())


@pytest.mark.parametrize("T,E,top,K_,N", [(1, 3, 1, 1024, 1), (1, 600, 2, 1032, 40), (5, 4, 3, 1536, 17), (16, 5, 2, 2048, 200), (16, 2, 2, 2056, 33), (17, 3, 2, 2048, 48),
                                          (32, 2, 1, 1024, 31), (32, 40, 4, 4096, 16), (9, 2, 1, 4096, 100)])
def test_experts_of_few_rows(K, T, E, top, K_, N):
    """Experts whose rows stay in registers, in all forms of their products, against float64: more experts than workgroups of a share and than
    workgroups, tiles of W that end inside one, K that leaves waves part of their steps.  The result is rounded to bfloat16 (2^-9 of it), the
    float sums before that are good to 2^-24 sqrt(K) of a sum of magnitude one, and a gate's activation passes on at most 1.1 times that: 2^-8 covers both.
    An infinite number in W reaches its own output alone."""
    g = torch.Generator().manual_seed(T * 31 + K_ + N)
    plan = K.moe_route(torch.randn((T, E), generator=g).to(DEV), E, top)
    perm, ids = plan.perm.cpu().long(), plan.ids.cpu().long().flatten()
    token, expert, weight = perm // top, ids[perm], plan.weights.cpu().flatten()[perm]
    x = torch.randn((T, K_), generator=g).to(BF16)
    w = (torch.randn((E, 2 * N, K_), generator=g) / math.sqrt(K_)).to(BF16)
    w[expert[0], 0, K_ - 1] = math.inf
    xd, wd = x.to(DEV), w.to(DEV)
    wp = wd[:, :N].contiguous()
    assert T <= K.MOE_FEW_TOKENS

    def product(rows, form):
        return torch.stack([w[e, :N if form == "plain" else 2 * N].to(F64) @ r for e, r in zip(expert.tolist(), rows.to(F64))])

    def glu(rows, limit):
        z = product(rows, "glu")
        a, b = z[:, :N], z[:, N:]
        if limit is None:
            return a * torch.sigmoid(a) * b
        a, b = a.clamp(max=limit), b.clamp(-limit, limit)
        return a * torch.sigmoid(1.702 * a) * (b + 1)

    rows = x[token]
    scaled = (rows.float() * weight[:, None]).to(BF16)
    order = rows.to(DEV)
    for got, want in ((K.moe_gemm(xd, wd, plan, True, act="silu", weighted=False), glu(rows, None)), (K.moe_gemm(xd, wd, plan, True, 0.8), glu(scaled, 0.8)),
                      (K.moe_gemm(order, wp, plan, False), product(rows, "plain")),
                      (K.moe_gemm(xd, wp, plan, False, gather=True, act="relu2"), product(rows, "plain").clamp(min=0) ** 2)):
        got = got.cpu()
        whole = torch.isfinite(want)
        assert whole.sum() >= want.numel() - 2 * T and torch.isfinite(got.float())[whole].all()
        torch.testing.assert_close(got.to(F64)[~whole], want[~whole], equal_nan=True)
        _close(torch.where(whole, got.to(F64), 0.0), torch.where(whole, want, 0.0), 2.0 ** -8)


@pytest.mark.parametrize("T,E,top,K_,N", [(1, 3, 1, 1024, 40), (16, 14, 2, 1536, 33), (16, 5, 2, 2048, 200), (7, 600, 2, 1032, 17), (32, 3, 2, 2056, 48), (32, 14, 2, 1280, 100),
                                          (32, 2, 2, 4096, 65), (12, 40, 4, 3848, 16)])
def test_experts_of_few_rows_give_the_bits_of_many(K, monkeypatch, T, E, top, K_, N):
    """A token's product by its expert in a step of few tokens and in one of more than the few-rows kernel takes, in every form: the same bits."""
    g = torch.Generator().manual_seed(T + E + K_)
    z, x = torch.randn((33, E), generator=g), torch.randn((33, K_), generator=g).to(BF16).to(DEV)
    w = (torch.randn((E, 2 * N, K_), generator=g) / math.sqrt(K_)).to(BF16).to(DEV)
    wp = w[:, :N].contiguous()
    assert T <= K.MOE_FEW_TOKENS < 33

    def pairs(tokens):
        """[tokens, top, outputs] of every form"""
        plan = K.moe_route(z[:tokens].to(DEV), E, top)
        place = plan.inv.long()
        rows = x[plan.perm.long() // top]
        return [y[place].view(tokens, top, -1) for y in (K.moe_gemm(x[:tokens], w, plan, True, act="silu", weighted=False), K.moe_gemm(x[:tokens], w, plan, True, 0.8),
                                                         K.moe_gemm(rows, wp, plan, False), K.moe_gemm(x[:tokens], wp, plan, False, gather=True, act="relu2"))]

    few = pairs(T)
    for a, b in zip(few, pairs(33)):
        assert torch.equal(a, b[:T])
    monkeypatch.setattr(K, "MOE_FEW_TOKENS", 0)
    for a, b in zip(few, pairs(T)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("M,N,K_,cut", [(1024, 2304, 2304, True), (1024, 2112, 2304, True), (2048, 1280, 1024, False), (2048, 1024, 1024, False), (1024, 6912, 2304, False),
                                        (2048, 4608, 4096, True), (255 * 128, 256, 8192, False), (255 * 128, 200, 32768, False), (2048, 4096, 4096, False), (65, 60000, 4096, False),
                                        (1, 1 << 20, 4, False), (65, 64, 1 << 20, True)])
def test_float32_cut_tiles_by_size_and_their_workspace(K, M, N, K_, cut):
    """Where two to three tiles of 64 x 64 a unit would run beyond one another the rule cuts, and no size asks for more than a slice's sums of every unit but one."""
    from infinilm_amd.csrc import lib
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    need = lib.load().ilm_gemm_f32_cut_ws(M, N, K_)
    assert 0 <= need <= (cus - 1) * 8 * 128 * 256
    assert cus != 256 or (need > 0) == cut


@pytest.mark.parametrize("tile,M,N,K_", [(1, 1100, 1220, 64), (1, 1990, 700, 128), (2, 2041, 1000, 64), (2, 4000, 330, 192), (3, 4000, 1100, 64), (1, 130, 2000, 64)])
def test_portion_product_walks_its_tiles_in_bands(K, tile, M, N, K_):
    """Products whose tiles are walked in bands of several rows of tiles, the last band lower than the others: every output once.  float sums of products of
    bfloat16 (2^-24 sqrt(K) of the norm of the addends) and one rounding to bfloat16, 2^-9: 2^-8 of the largest."""
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K_), generator=g).to(BF16).to(DEV), torch.randn((N, K_), generator=g).to(BF16).to(DEV)
    out = torch.full((M, N), math.nan, dtype=BF16, device=DEV)
    K.portion_gemm(x, w, None, out, tile)
    want = x.to(F64) @ w.to(F64).T
    assert float((out.to(F64) - want).abs().max()) < 2.0 ** -8 * float(want.abs().max())


@pytest.mark.parametrize("n", [1, 16, 17, 64, 65, 192, 193])
@pytest.mark.parametrize("V", [3000, 50000])
def test_sampling_with_the_rows_settings_in_the_launch(K, n, V):
    """Settings that travel with the launch, for every size of that form and the first beyond it, and the sampler that uses it: the tokens of settings in
    device memory, by one workgroup a row and in chunks; launched twice and recorded, so that no launch sees another's."""
    from array import array
    from infinilm_amd.sampling import Sampler, SamplingParams
    from infinilm_amd.sampling.sampler import uniforms_for
    g = torch.Generator().manual_seed(n + V)
    logits = (2.0 * torch.randn((n, V), generator=g)).to(DEV)
    settings = [(0.5 + i % 5 * 0.2, (0, 1, 20, 400)[i % 4], (1.0, 0.9, 0.3)[i % 3], 1000 + i * (1 << 40), i) for i in range(n)]
    t, k, p, keys, index = (list(x) for x in zip(*settings))
    prm = torch.cat([torch.tensor(t), torch.tensor(k, dtype=torch.int32).view(torch.float32), torch.tensor(p),
                     torch.from_numpy(uniforms_for([9] * n, keys, index))]).to(DEV)
    want = K.sample_packed(logits, prm)
    if n <= K.SAMPLE_HOST_ROWS:
        args = (array("f", t), array("i", k), array("f", p))
        one = K.sample_host(logits, *args, None, 9, array("Q", keys), array("Q", index))
        other = K.sample_host(logits, array("f", [1.0] * n), array("i", [1] * n), args[2], array("Q", [3] * n), 0, array("Q", keys), array("Q", index))
        assert torch.equal(one, want) and torch.equal(other, K.argmax(logits))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            rec = K.sample_host(logits, *args, array("Q", [9] * n), 0, array("Q", keys), array("Q", index))
        args[0][0] = 77.0
        for _ in range(3):
            rec.fill_(-1)
            graph.replay()
            assert torch.equal(rec, want)
    rows = [(SamplingParams(temperature=a, top_k=b, top_p=c), d, e) for a, b, c, d, e in settings]
    assert torch.equal(Sampler(9).sample_device(logits, rows), want)


@pytest.mark.parametrize("M,N,K_", [(1100, 2050, 64), (700, 3072, 192), (700, 2048, 320)])
def test_portion_gate_and_up_beyond_two_tiles_a_unit(K, M, N, K_):
    """Two stages in LDS instead of three, with one stage of K, three and five, against the product and the activation apart: the same bits."""
    g = torch.Generator().manual_seed(M + N + K_)
    x, w = torch.randn((M, K_), generator=g).to(BF16).to(DEV), torch.randn((2 * N, K_), generator=g).to(BF16).to(DEV)
    assert -(-M // 64) * -(-N // 64) > 2 * K._num_cus(torch.device(DEV)) or N == 2048
    got = K.portion_glu(x, w, None, "silu", 1)
    assert torch.equal(got, K.swiglu(K.portion_gemm(x, w, None, torch.empty((M, 2 * N), dtype=BF16, device=DEV), 1), "silu"))


@pytest.mark.parametrize("M,I,K_,act", [(65, 31, 36, "silu"), (127, 128, 260, "gelu_tanh"), (129, 515, 132, "silu"), (300, 257, 1028, "silu"), (1100, 4101, 132, "gelu_tanh")])
@pytest.mark.parametrize("odd", [False, True])
def test_gemm_float32_tiles_with_the_activation_in_their_epilogue(K, M, I, K_, act, odd):
    """Bit for bit the projection and the activation kernel one after the other, in whole tiles and in cut ones, with sums that the pieces cannot give in
    the gate, in up and in both, and a bias; and where the rule takes them."""
    from infinilm_amd.csrc import lib
    L = lib.load()
    g = torch.Generator().manual_seed(M + I + odd)
    x, w, b = torch.randn((M, K_), generator=g), torch.randn((2 * I, K_), generator=g) * 0.2, torch.randn((2 * I,), generator=g)
    if odd:
        x[M // 3, 3], x[M // 2, K_ - 1], x[M - 1] = math.inf, math.nan, x[M - 1] * 2.0 ** -80
        w[5, 7], w[I + 9, 8], w[I - 1, 9], w[2 * I - 1, 9] = math.inf, -math.inf, math.inf, -math.inf
        w[I // 2, :2], w[I, :2], x[0, :2] = torch.tensor([3e38, -3e38]), torch.tensor([3e38, -3e38]), torch.tensor([3.0, 3.0])
    x, w, b = x.to(DEV), w.to(DEV), b.to(DEV)
    stream = torch.cuda.current_stream().cuda_stream
    for bias in (None, b):
        want = K.swiglu(K.gemm(x, w, bias), act)
        assert not odd or not torch.isfinite(want).all()
        ws = torch.empty(((-(-M // 128)) * (-(-I // 128)) * 8 * 128 * 256,), device=DEV)
        for cut in (False, True):
            got = torch.full((M, I), 7.0, device=DEV)
            assert L.ilm_gemm_f32_glu_tile(got.data_ptr(), x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), M, I, K_, K_, K_, I,
                                           K.glu_code(act), ws.data_ptr() if cut else None, ws.numel() if cut else 0, stream) == 0
            _same(got, want)
        ruled = K.gateup_glu_f32(x, w, bias, act)
        assert (ruled is None) == (not L.ilm_gemm_f32_glu_tile_ok(M, I, K_))
        if ruled is not None:
            _same(ruled, want)


def test_gemm_float32_tiles_with_the_activation_are_taken_for_large_projections(K):
    """A whole number of rounds over the chip, and one that leaves tiles to be cut."""
    for M, K_ in ((512, 256), (700, 4096)):
        x, w = _rand((M, K_), 1).to(DEV), _rand((2 * 8192, K_), 2, scale=0.1).to(DEV)
        _same(K.gateup_glu_f32(x, w, None), K.swiglu(K.gemm(x, w)))
