"""The rules by which sizes choose a kernel, at the sizes where both sides were measured; no GPU."""
import pytest
import torch

from infinilm_amd import kernels as K

DEV = torch.device("cuda", 0)


@pytest.fixture(autouse=True)
def chip(monkeypatch):
    monkeypatch.setattr(K, "_num_cus", lambda device: 256)


@pytest.mark.parametrize("M,N,k,span", [(8, 1024, 4096, 1024), (16, 8192, 8192, 1024), (1, 4096, 4608, 1024), (8, 1023, 8192, 4096), (8, 4096, 8200, 4096),
                                        (17, 4096, 4096, 4096), (8, 8200, 4096, 4096), (1, 12288, 2048, 4096), (8, 12288, 8192, 4096),
                                        (16, 32768, 5120, 4096)])
def test_parts_of_a_few_rows_product(M, N, k, span):
    assert K._few_span(M, N, k) == span


@pytest.mark.parametrize("keys,pairs,d,reach,cut", [
    (500, 512, 64, 0, (512, 1)), (300, 256, 64, 0, (384, 1)), (1900, 512, 64, 0, (2048, 1)), (3800, 512, 64, 0, (2048, 2)),   # whole contexts
    (3800, 96, 64, 0, (512, 8)), (3800, 96, 64, 256, (1024, 4)), (3800, 96, 64, -256, (1024, 4)), (3800, 96, 64, 1024, (512, 8)),  # and windows
    (8000, 512, 64, 1024, (8192, 1)), (500, 128, 128, 0, (256, 2)), (500, 128, 128, 256, (384, 2)), (1900, 64, 64, 0, (128, 15)),
    (4096, 16, 128, 0, (256, 16)), (4096, 128, 128, 0, (1024, 4))])
def test_chunks_of_the_decode_attention(keys, pairs, d, reach, cut):
    span, chunks = K.attention_chunks(keys, 64, pairs, DEV, d, reach)
    assert (span, chunks) == cut and span * (chunks - 1) < keys <= span * chunks


@pytest.mark.parametrize("M,N,k,tile", [
    (2048, 1024, 1024, 2), (300, 1024, 1024, 1), (65, 8192, 1024, 1), (600, 4096, 2048, 3), (2048, 1024, 4096, 2), (700, 1024, 4096, 1),
    (2048, 1024, 1000, 0), (2048, 2048, 8192, 0), (700, 8192, 1024, 0), (300, 1024, 4096, 0),        # stages, a long K, two rounds, half of the units
    (65, 512, 1024, 1), (65, 512, 2048, 0), (512, 256, 1536, 1), (65, 1024, 2048, 1),                # an eighth
    (2048, 512, 2048, 0), (2048, 512, 1024, 1), (1000, 512, 2048, 1), (8192, 512, 1024, 0), (8192, 512, 512, 3), (2048, 768, 3072, 0), (2048, 768, 1536, 2),
    (1000, 16, 512, 0), (1000, 16, 256, 1), (128, 16, 512, 1), (128, 16, 1024, 0),                   # few outputs
    (923, 3853, 2304, 0), (137, 8717, 640, 0), (249, 2381, 2880, 1)])                                # odd rows
def test_portions_products(M, N, k, tile):
    assert K._portion_tile("plain", M, N, k, DEV) == tile


@pytest.mark.parametrize("M,N,k,tile", [
    (1024, 1280, 1024, 1), (256, 4608, 4096, 1), (300, 4608, 4096, 2), (2048, 1280, 1024, 2), (2041, 1280, 2048, 2), (256, 6912, 2304, 2),
    (512, 4608, 4096, 0), (505, 4608, 3584, 0), (300, 6144, 4096, 0), (1400, 1536, 512, 0), (1280, 1536, 512, 2), (2048, 6912, 2304, 0)])
def test_portions_projections_with_rotation(M, N, k, tile):
    assert K._portion_tile("rope", M, N, k, DEV) == tile


@pytest.mark.parametrize("M,N,k,tile", [
    (300, 8192, 1024, 1), (700, 8192, 1024, 1), (1000, 8192, 1024, 4), (2048, 8192, 1024, 5), (300, 16384, 768, 1), (500, 16384, 768, 4),
    (65, 1024, 1024, 0), (130, 1536, 768, 1), (33, 512, 1024, 0), (200, 1024, 1024, 1), (65, 2048, 1024, 1), (65, 512, 512, 1), (400, 12288, 2048, 0)])
def test_portions_gate_and_up(M, N, k, tile):
    assert K._portion_tile("glu", M, N, k, DEV) == tile


@pytest.mark.parametrize("n,V,k,one", [
    (1, 32768, 224, True), (64, 73448, 50, True), (5, 49152, 224, True), (1, 65536, 128, True), (1, 65536, 192, False), (2, 73448, 128, True),
    (8, 73448, 160, False), (4, 98000, 96, True), (1, 98000, 112, False), (5, 122753, 50, True), (1, 122753, 96, True), (1, 152064, 16, False), (5, 122753, 100, False), (1, 122753, 200, False),
    (8, 152064, 64, False), (16, 122753, 160, True), (12, 152064, 160, False), (32, 122753, 224, True), (64, 152064, 224, True), (64, 152064, 225, False)])
def test_route_of_a_small_top_k(n, V, k, one):
    assert K.sample_one_reading(n, V, k) == one


@pytest.mark.parametrize("M,k,taken", [(1, 2048, True), (2, 1024, True), (8, 256, True), (1, 3328, True), (1, 4096, True), (1, 2304, False), (1, 3072, False),
                                       (2, 2048, False), (1, 1000, False), (1, 4352, False), (9, 256, False)])
def test_rows_that_the_projection_forms(M, k, taken):
    assert K._qkv_sum_rows(M, k) == taken


@pytest.mark.parametrize("M,k,N,parts,taken", [(1, 2048, 6144, 8, True), (2, 1024, 1280, 8, True), (2, 1024, 3072, 4, True), (2, 1024, 3072, 8, False),
                                               (4, 512, 4608, 5, False), (8, 256, 6144, 8, True), (4, 256, 6144, 8, True)])
def test_parts_that_the_projection_sums(M, k, N, parts, taken):
    assert K._qkv_sum_parts(M, k, N, parts) == taken


@pytest.mark.parametrize("T,one", [(1, True), (16, True), (17, False), (64, False)])
def test_experts_are_chosen_and_ordered_in_one_kernel_for_few_tokens(monkeypatch, T, one):
    from types import SimpleNamespace

    called = []
    monkeypatch.setattr(K, "_dev", lambda *a: None)
    monkeypatch.setattr(K, "_stream", lambda: 0)
    monkeypatch.setattr(K, "_lib", lambda: SimpleNamespace(ilm_moe_plan_few_ok=lambda *a: 1, ilm_moe_tile_rows=lambda: 16, ilm_moe_big_tile_rows=lambda: 128))
    monkeypatch.setattr(K, "_run", lambda name, *a, **k: called.append(name))
    K.moe_route(torch.zeros(T, 16), 16, 2, softmax=True, groups=4, keep=2, correction=torch.zeros(16), normalise=True)
    assert called == (["ilm_moe_plan_few"] if one else ["ilm_moe_route_groups", "ilm_moe_sort"])


@pytest.mark.parametrize("T,tiles,singles,nh,nkv,d,bound,how", [
    (768, 96 + 64, 64, 32, 2, 128, 16384, (True, True, True)), (740, 92, 5, 32, 2, 128, 16000, (True, True, True)),     # a recorded step's lists, an eager one's
    (2048, 256 + 64, 64, 32, 2, 128, 16384, (True, False, True)), (2048, 256, 0, 32, 2, 128, 2048, (True, False, False)),
    (1200, 13, 1100, 32, 2, 128, 4096, (False, False, False)),                                                          # a short portion beside many tokens
    (2400, 163, 1100, 32, 2, 128, 4096, (True, False, False)), (300, 38, 3, 36, 36, 64, 2048, (True, True, True)), (300, 38, 60, 36, 36, 64, 2048, (True, True, False)),
    (300, 38, 3, 36, 36, 64, 128, (True, False, False)), (300, 38, 3, 16, 2, 80, 2048, (False, False, True)), (64, 0, 0, 32, 2, 128, 4096, (False, False, True)),
    (2048, 256, 0, 16, 2, 128, 2048, (True, True, False)), (2048, 256, 0, 16, 2, 128, 2049, (True, False, False)), (1536, 192, 0, 16, 2, 128, 32768, (True, True, False)),
    (1537, 193, 0, 16, 2, 128, 32768, (True, False, False)), (1024, 0, 0, 32, 2, 128, 32768, (False, False, True)),
    (256, 32, 0, 32, 2, 128, 4096, (False, False, True)), (257, 33, 0, 32, 2, 128, 4096, (True, True, False))])
def test_32_bit_attention_of_tiles_and_single_rows(T, tiles, singles, nh, nkv, d, bound, how):
    """Each list is cut into chunks, or not, by its own length."""
    got = K.f32_attention(T, tiles, singles, nh, nkv, d, 64, bound)
    assert (got.tiled, got.split_tiles, got.split_rows) == how and got.chunks == -(-bound // K.F32_ATTN_CHUNK)


@pytest.mark.parametrize("T,tiles,singles,nh,nkv,d,bound", [(1536, 192, 0, 16, 2, 128, 32768), (768, 96, 0, 32, 2, 128, 32768), (300, 38, 40, 36, 36, 64, 32768),
                                                            (1000, 0, 0, 32, 2, 128, 131072), (8, 1, 0, 128, 8, 256, 1 << 20), (512, 64 + 64, 64, 32, 2, 128, 65536)])
def test_32_bit_attention_holds_a_bounded_workspace(T, tiles, singles, nh, nkv, d, bound):
    """Long contexts whose tiles or tokens are cut into chunks: partial results of at most 1 GiB at once, or of eight tokens."""
    how = K.f32_attention(T, tiles, singles, nh, nkv, d, 64, bound)
    assert how.split_tiles or how.split_rows
    row = 4 * nh * how.chunks * (d + 4)
    assert how.most == 8 or how.most * row <= 1 << 30
    for n, most in ((tiles, how.most // K.ATT_TILE_TOKENS), (singles or T, how.most)):
        runs = K._runs(n, most) if n else []
        assert all(0 < m <= most for _, m in runs) and [a for a, _ in runs] == [sum(m for _, m in runs[:i]) for i in range(len(runs))] and sum(m for _, m in runs) == n


def test_32_bit_attention_takes_any_page_and_any_number_of_tiles():
    """Pages beyond the tile kernel's 32-bit offsets go to the other one, tiles beyond a grid to several launches."""
    assert K.f32_attention(2048, 256, 0, 32, 2, 128, (1 << 21) - 16, 2048).tiled and not K.f32_attention(2048, 256, 0, 32, 2, 128, 1 << 21, 2048).tiled
    how = K.f32_attention(1 << 20, 1 << 17, 0, 4, 4, 64, 64, 2048)
    assert how.tiled and how.most_tiles == 65535 and [n for _, n in K._runs(1 << 17, how.most_tiles)] == [43690, 43691, 43691]
