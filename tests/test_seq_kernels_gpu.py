"""Each kernel of ``csrc/kernels/seq`` against the plain PyTorch op of the same name
(``ops/torch_seq.py``, fp32 arithmetic), on shapes that exercise every tile path, tail and batch form:
GEMMs (64 / 128 / 256 tiles, the skinny decode kernel, K tails, column-slice operands, strided batch,
row groups), group norm, activations, K/V store, both attention kernels over paged keys (chunks, windows,
carried positions, head sizes on and off the matrix-core path), convolution and both scans with carried
state in scattered slots, routing."""
import math

import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not gpu_available():
        pytest.skip("no GPU")
    from flexible_llm_sharding_amd.ops.hip_seq import HipSeqOps
    from flexible_llm_sharding_amd.ops.torch_seq import TorchSeqOps
    return HipSeqOps(), TorchSeqOps()


def close(a, b, tol):
    a, b = a.float().cpu(), b.float().cpu()
    e = (a - b).abs().max().item() / (b.abs().max().item() + 1e-9)
    assert e < tol, e


def meta_of(lens, pos0, dev, ps=16, seed=0):
    rng = np.random.default_rng(seed)
    B = len(lens)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    seq = np.repeat(np.arange(B), lens).astype(np.int32)
    pos = np.concatenate([np.arange(p, p + n) for p, n in zip(pos0, lens)]).astype(np.int32)
    npg = [-(-(p + n) // ps) for p, n in zip(pos0, lens)]
    tab = np.full((B, max(npg)), -1, np.int32)
    perm = rng.permutation(sum(npg) + 5)
    k = 0
    for b in range(B):
        for j in range(npg[b]):
            tab[b, j] = perm[k]
            k += 1
    slot = rng.permutation(B + 3)[:B].astype(np.int32)
    kvs = (tab[seq, pos // ps].astype(np.int64) * ps + pos % ps).astype(np.int32)
    m = dict(tok_seq=seq, tok_pos=pos, cu=cu, pos0=np.array(pos0, np.int32), slot=slot, page_table=tab, kv_slot=kvs)
    md = {k: torch.from_numpy(v).to(dev) for k, v in m.items()}
    md.update(n_seqs=B, cu_host=cu, pos0_host=np.array(pos0), max_rows=max(lens))
    if max(lens) >= 16:
        md["q_tiles"] = torch.tensor([(a + o, min(128, b - a - o)) for a, b in zip(cu[:-1], cu[1:])
                                      for o in range(0, b - a, 128)], dtype=torch.int32, device=dev)
        md["tile_cu"] = torch.tensor(np.concatenate([[0], np.cumsum([-(-int(n) // 128) for n in lens])]), dtype=torch.int32,
                                     device=dev)
    return md, sum(npg) + 5, B + 3


DTYPES = [(torch.float32, 2e-5), (torch.bfloat16, 2e-2)]
DEV = "cuda:0"


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("M,N,K", [(5, 70, 33), (130, 192, 256), (64, 64, 64), (1, 454, 256), (300, 200, 454), (257, 129, 72),
                                   (4100, 4200, 136), (8, 200, 512), (32, 64, 72), (17, 100, 2056), (3, 4096, 1024)])
def test_matmul(ops, cdt, tol, M, N, K):
    H, R = ops
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K, device=DEV).to(cdt)
    w = torch.randn(N, K, device=DEV).to(cdt)
    b = torch.randn(N, device=DEV)
    close(H.matmul_nt(a, w, b), R.matmul_nt(a, w, b), 1e-5)
    act = torch.tensor([0.4, -0.3], device=DEV)                     # activation and rounding in the epilogue
    close(H.matmul_nt(a, w, b, xielu=act, out_dtype=cdt), R.matmul_nt(a, w, b, xielu=act, out_dtype=cdt), tol)
    af = torch.randn(M, K + 8, device=DEV)[:, 4:4 + K]             # fp32 rows, a column slice: rounded on the way in
    close(H.matmul_nt(af, w), R.matmul_nt(af.to(cdt), w), 1e-5)


# sizes that take each bf16 tile of gemm_tile.hip (256 x 256, 128 x 128 twice, 64 x 128, 64 x 64, 32 x 64, 32 x 32, 192 and 128 x 256) for the plain
# product, with rows and columns past a tile's end and odd numbers of 64-wide K tiles (which tile is asserted in test_every_tile).  fp32 sums of bf16 products: 1e-5; rounded to bf16: half a
# unit in the last place of the largest value (2^-9) and the other side's sum
@pytest.mark.parametrize("M,N,K", [(2100, 4100, 64), (4100, 4100, 192), (1030, 4000, 64), (1024, 3900, 320), (1000, 2000, 320), (257, 2020, 320),
                                   (200, 2000, 1088), (65, 132, 448), (4000, 4092, 320), (2500, 4100, 320), (3000, 4092, 256), (2000, 4000, 1984), (1025, 7000, 1088)])
def test_matmul_tiles(ops, M, N, K):
    H, R = ops
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K + 8, device=DEV).bfloat16()[:, 8:]
    w = (0.1 * torch.randn(N, K, device=DEV)).bfloat16()
    b = torch.randn(N, device=DEV)
    close(H.matmul_nt(a, w, b), R.matmul_nt(a, w, b), 1e-5)
    close(H.matmul_nt(a, w, out_dtype=torch.bfloat16), R.matmul_nt(a, w, out_dtype=torch.bfloat16), 2 ** -8)
    act = torch.tensor([0.4, -0.3], device=DEV)
    close(H.matmul_nt(a, w, b, xielu=act), R.matmul_nt(a, w, b, xielu=act), 1e-5)
    rates = torch.tensor([0.2, -0.5, 0.1, 0.3], device=DEV)
    close(H.matmul_nt(a, w, b, decay=rates), R.matmul_nt(a, w, b, decay=rates), 1e-5)
    E = 5                                                           # row groups, empty ones among them
    offs = torch.tensor([0, 0, M // 2, M // 2 + 1, M, M], dtype=torch.int32, device=DEV)
    wg = (0.1 * torch.randn(E, N, K, device=DEV)).bfloat16()
    close(H.grouped_matmul_nt(a, wg, offs), R.grouped_matmul_nt(a, wg, offs), 1e-5)


# the same for fp32 operands and for fp32 rows against bf16 weights, blocks of a strided batch (their tiles one by one: test_every_tile)
@pytest.mark.parametrize("M,N,K", [(4000, 2052, 96), (1300, 2500, 160), (520, 2052, 224), (260, 2052, 288), (130, 1028, 352), (40, 132, 416)])
def test_matmul_tiles_fp32_rows(ops, M, N, K):
    H, R = ops
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K + 4, device=DEV)[:, 4:]
    w = 0.1 * torch.randn(N, K, device=DEV)
    b = torch.randn(N, device=DEV)
    want = (a.double() @ w.double().t() + b.double()).float()
    close(H.matmul_nt(a, w, b), want, 1e-5)
    kt = -(-K // 64) * 64
    a, w = torch.randn(M, kt, device=DEV), (0.1 * torch.randn(N, kt, device=DEV)).bfloat16()
    close(H.matmul_nt(a, w, b), R.matmul_nt(a.bfloat16(), w, b), 1e-5)
    u, wg, bg = torch.randn(M, 192, device=DEV), torch.randn(6, 64, 64, device=DEV).bfloat16(), torch.randn(6 * 64, device=DEV)
    close(H.block_linear(u, wg, bg, 3, torch.bfloat16), R.block_linear(u, wg, bg, 3, torch.bfloat16), 1e-5)


# gated products ([gate; up] rows of W, the gate in the epilogue): few rows, some of the tiles (each of them: test_every_tile), experts with
# gathered rows, and rows no tile takes (K = 100: the product and the gate as two kernels)
@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("M,I,K", [(5, 40, 64), (23, 100, 200), (70, 1028, 192), (300, 1028, 64), (1030, 2052, 64), (2100, 2052, 64), (20, 24, 100)])
def test_gated_matmul(ops, cdt, tol, M, I, K):
    H, R = ops
    torch.manual_seed(M + I + K)
    a, w = torch.randn(M, K, device=DEV).to(cdt), (0.2 * torch.randn(2 * I, K, device=DEV)).to(cdt)
    for act, lim in (("silu", 0.0), ("gelu_tanh", 0.0), ("clamped", 0.7)):
        close(H.gated_matmul_nt(a, w, cdt, act, lim), R.gated_matmul_nt(a, w, cdt, act, lim), tol)
        close(H.gated_matmul_nt(a, w, torch.float32, act, lim), R.gated_matmul_nt(a, w, torch.float32, act, lim), 2e-5)
    E, n = 5, 2 * M                                                 # two places per row of a, the last ones in no expert's range
    rows = torch.randperm(n, device=DEV).to(torch.int32) // 2
    offs = torch.tensor([0, 0, M, M + 1, n - 2, n - 2], dtype=torch.int32, device=DEV)
    wg = (0.2 * torch.randn(E, 2 * I, K, device=DEV)).to(cdt)
    close(H.gated_matmul_nt(a, wg, cdt, offs=offs, rows=rows)[:n - 2], R.gated_matmul_nt(a, wg, cdt, offs=offs, rows=rows)[:n - 2], tol)
    z = H.matmul_nt(a, w, softcap=3.0)
    close(z, R.matmul_nt(a, w, softcap=3.0), 2e-5)
    close(H.matmul_nt(a, w, scale=0.3), R.matmul_nt(a, w, scale=0.3), 1e-5)
    wide = torch.cat([z, z[:, :1]], 1)[:, :2 * I]                   # (a row stride that is no multiple of four)
    for t in (z, wide):
        assert torch.equal(H.argmax_f32(t), t.argmax(1).to(torch.int32))


# every tile of gemm_tile.hip by the index in its table (the library says which one a product takes, so a changed rule shows here): plain with a
# bias, an activation and bf16 results; gated; row groups, empty and of one row among them; gated row groups from gathered rows.  Rows and
# columns past a tile's end, odd numbers of K tiles.  Sums as in test_matmul_tiles, bf16 operands against fp64 of their products
EVERY_TILE = [("bf16", v, p, g) for v, (p, g) in enumerate([
    ((8200, 1304, 192), (2500, 4104, 192)), ((390, 8200, 192), (130, 8200, 192)), ((200, 8200, 192), (200, 5128, 192)), ((65, 8200, 192), (130, 4104, 192)),
    ((65, 72, 192), (130, 72, 192)), ((65, 3080, 448), (130, 1032, 448)), ((65, 72, 320), (130, 72, 320)), ((900, 8200, 192), (700, 8200, 192)),
    ((390, 8200, 1088), (200, 8200, 1088))])]
EVERY_TILE += [("mixed", v, p, g) for v, (p, g) in enumerate([
    ((200, 8200, 192), (1700, 1544, 192)), ((65, 8200, 1088), (130, 3080, 1088)), ((65, 3080, 192), (130, 1032, 192)), ((65, 8200, 192), (130, 3080, 192)),
    ((65, 72, 192), (130, 72, 192))])]
EVERY_TILE += [("fp32", v, p, g) for v, (p, g) in enumerate([
    ((8200, 392, 96), (257, 8200, 96)), ((8200, 136, 64), (200, 5128, 96)), ((65, 8200, 96), (130, 4104, 96)), ((4100, 72, 96), (130, 2056, 96)),
    ((65, 3080, 96), (130, 1032, 96)), ((65, 72, 96), (130, 72, 96))])]


@pytest.mark.parametrize("types,tile,plain,grouped", EVERY_TILE)
def test_every_tile(ops, types, tile, plain, grouped):
    H, _ = ops
    ta, tw = {"bf16": (torch.bfloat16, torch.bfloat16), "mixed": (torch.float32, torch.bfloat16), "fp32": (torch.float32, torch.float32)}[types]
    code, E = lambda t: int(t == torch.bfloat16), 6
    gated = (types, tile) not in (("bf16", 6), ("mixed", 4), ("fp32", 5))           # (32-column tiles hold one half of a gated column)
    for (M, N, K), groups in ((plain, 1), (grouped, E)):
        for g in (0, 1)[:1 + gated]:
            assert H.k.fls_seq_gemm_tile_of(code(ta), code(tw), M, N, K, groups, int(groups > 1), g) == tile
    f64 = lambda t: (t.to(tw) if types == "mixed" else t).double()                  # (fp32 rows are rounded to bf16 weights)
    M, N, K = plain
    torch.manual_seed(M + N + K)
    a, w, b = torch.randn(M, K, device=DEV).to(ta), (0.1 * torch.randn(N, K, device=DEV)).to(tw), torch.randn(N, device=DEV)
    z = f64(a) @ w.double().t()
    close(H.matmul_nt(a, w, b), z + b, 1e-5)
    close(H.matmul_nt(a, w, b, relu2=True, out_dtype=torch.bfloat16), torch.relu(z + b).square(), 2 ** -8)
    silu = lambda y: torch.nn.functional.silu(y[..., :y.shape[-1] // 2]) * y[..., y.shape[-1] // 2:]
    if gated:
        close(H.gated_matmul_nt(a, w, torch.float32), silu(z), 2e-5)
        close(H.gated_matmul_nt(a, w, torch.bfloat16), silu(z), 2 ** -8)
    M, N, K = grouped
    sizes = [0, M // 2, 1, M - M // 2 - 1 - 3, 0, 3]
    offs = torch.tensor(np.cumsum([0] + sizes), dtype=torch.int32, device=DEV)
    a, w = torch.randn(M, K, device=DEV).to(ta), (0.1 * torch.randn(E, N, K, device=DEV)).to(tw)
    y = lambda x: torch.cat([f64(x[offs[e]:offs[e + 1]]) @ w[e].double().t() for e in range(E)])
    close(H.grouped_matmul_nt(a, w, offs), y(a), 1e-5)
    if gated:
        rows, few = torch.randperm(M, device=DEV).to(torch.int32) // 2, a[:(M + 1) // 2]        # (two places per row)
        for out, tol in ((torch.float32, 2e-5), (torch.bfloat16, 2 ** -8)):
            close(H.gated_matmul_nt(few, w, out, offs=offs, rows=rows), silu(y(few[rows.long()])), tol)


# 64 x 128 tiles, two blocks a CU: long plain and gated products, rows and columns past the last tile's end, an odd number of K tiles.
# fp32 sums of up to 2,048 products of the same bf16 operands: 1e-5 as in test_matmul_tiles
@pytest.mark.parametrize("M,N,K", [(1000, 4040, 1216), (1024, 4096, 2048), (511, 7688, 1152)])
def test_two_blocks_a_unit(ops, M, N, K):
    H, _ = ops
    assert [H.k.fls_seq_gemm_tile_of(1, 1, M, N, K, 1, 0, g) for g in (0, 1)] == [9, 9]
    torch.manual_seed(M + N + K)
    a, w = torch.randn(M, K, device=DEV).bfloat16(), (0.1 * torch.randn(N, K, device=DEV)).bfloat16()
    z = a.double() @ w.double().t()
    close(H.matmul_nt(a, w), z, 1e-5)
    close(H.gated_matmul_nt(a, w, torch.float32), torch.nn.functional.silu(z[:, :N // 2]) * z[:, N // 2:], 2e-5)


# 256-column tiles of 160, 224, 288 and 320 rows, whose row groups leave an odd one over and, in the two tallest, are partly held apart from the rest:
# long plain and gated products, both result types, rows and columns past the last tile's end, an odd number of K tiles; tolerances as above
@pytest.mark.parametrize("tile,M,N,K", [(10, 776, 9352, 1216), (11, 1169, 9264, 1216), (12, 1540, 9416, 1216), (13, 1731, 9360, 1216), (13, 2560, 8192, 1152)])
def test_tile_heights(ops, tile, M, N, K):
    H, _ = ops
    assert [H.k.fls_seq_gemm_tile_of(1, 1, M, N, K, 1, 0, g) for g in (0, 1)] == [tile, tile]
    torch.manual_seed(M + N + K)
    a, w, b = torch.randn(M, K, device=DEV).bfloat16(), (0.1 * torch.randn(N, K, device=DEV)).bfloat16(), torch.randn(N, device=DEV)
    z = a.double() @ w.double().t()
    close(H.matmul_nt(a, w, b), z + b, 1e-5)
    close(H.matmul_nt(a, w, b, relu2=True, out_dtype=torch.bfloat16), torch.relu(z + b).square(), 2 ** -8)
    gate = torch.nn.functional.silu(z[:, :N // 2]) * z[:, N // 2:]
    close(H.gated_matmul_nt(a, w, torch.float32), gate, 2e-5)
    close(H.gated_matmul_nt(a, w, torch.bfloat16), gate, 2 ** -8)


# few rows per group, one group of more than the 16 that a pass over its weights takes, empty groups, a K tail
@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("K", [64, 200])
def test_grouped_few_rows(ops, cdt, tol, K):
    H, R = ops
    torch.manual_seed(K)
    offs = torch.tensor([0, 0, 30, 31, 37, 37], dtype=torch.int32, device=DEV)
    a, w = torch.randn(37, K, device=DEV).to(cdt), torch.randn(5, 100, K, device=DEV).to(cdt)
    close(H.grouped_matmul_nt(a, w, offs), R.grouped_matmul_nt(a, w, offs), 1e-5)


# more column blocks than the chip has CUs over all groups (four waves a block, twice the steps in flight): whole chunks of them, what is left
# and a K tail, plain and gated, rows as they are and gathered
@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("K", [64, 200, 1024, 1096])
def test_grouped_few_rows_many_blocks(ops, cdt, tol, K):
    H, R = ops
    torch.manual_seed(K)
    sizes = [0, 1, 0, 17, 2] + [0, 1] * 18 + [3]
    M, E, N = sum(sizes), len(sizes), 112
    offs = torch.tensor([0] + sizes).cumsum(0).int().to(DEV)
    a, w = torch.randn(M, K, device=DEV).to(cdt), torch.randn(E, 2 * N, K, device=DEV).to(cdt)
    close(H.grouped_matmul_nt(a, w, offs), R.grouped_matmul_nt(a, w, offs), 1e-5)
    close(H.grouped_matmul_nt(a, w[:, :N].contiguous(), offs), R.grouped_matmul_nt(a, w[:, :N].contiguous(), offs), 1e-5)
    for rows in (None, torch.randperm(M).int().to(DEV)):
        close(H.gated_matmul_nt(a, w, torch.float32, offs=offs, rows=rows), R.gated_matmul_nt(a, w, torch.float32, offs=offs, rows=rows), 1e-5)


# decays of -200 .. 200 through an identity product, and of infinities and NaN from the bias, in a few-row block and a tile.  The product of rate and softplus is good to a
# unit of its last place, whose share of the result is that place itself, up to 88: 88 x 2^-24, and a unit each for the exponential and the sum
@pytest.mark.parametrize("T", [5, 300])
def test_decay_values(ops, T):
    H, _ = ops
    torch.manual_seed(T)
    z = (torch.randn(T, 128, device=DEV) * 10 ** (torch.rand(T, 128, device=DEV) * 4 - 2)).clamp(-200, 200).bfloat16()
    z[0, :2] = torch.tensor([0.0, -0.0], device=DEV)
    rates = torch.tensor([-4.0, 0.0, 1.0, 2.8], device=DEV)
    eye = torch.eye(128, device=DEV).bfloat16()
    y = H.matmul_nt(z, eye, torch.zeros(128, device=DEV), decay=rates)
    want = torch.exp(-rates.double().exp().repeat_interleave(32) * torch.nn.functional.softplus(z.double(), threshold=1000))
    assert ((y.double() - want).abs() <= 90 * 2 ** -24 * want + 2.0 ** -126).all()
    b = torch.zeros(128, device=DEV)
    b[:3] = torch.tensor([float("inf"), float("-inf"), float("nan")], device=DEV)
    y = H.matmul_nt(z, eye, b, decay=rates)
    assert (y[:, 0] == 0).all() and (y[:, 1] == 1).all() and y[:, 2].isnan().all()


# decays at the ends of fp32, as exp(-exp(act) softplus(z)) has them: results below 2^-126 (within a unit of their last place beside the share above), rates of zero, of
# next to nothing under a huge z, and infinite ones, each with the bias's infinities
@pytest.mark.parametrize("T", [5, 300])
def test_decay_edges(ops, T):
    H, _ = ops
    inf = float("inf")
    eye, zero = torch.eye(128, device=DEV).bfloat16(), torch.zeros(T, 128, device=DEV).bfloat16()
    z = torch.linspace(80, 110, T * 128, device=DEV).view(T, 128).bfloat16()
    y = H.matmul_nt(z, eye, torch.zeros(128, device=DEV), decay=torch.zeros(4, device=DEV))
    want = torch.exp(-z.double())
    assert (want < 2.0 ** -126).any() and (want > 2.0 ** -126).any()
    assert ((y.double() - want).abs() <= 110 * 2 ** -24 * want + 2.0 ** -149).all()
    b = torch.tensor([inf, -inf, float("nan"), 1e33, 3e38, 0.0, -85.0, -60.0], device=DEV).repeat(16)
    for act, want in ((-inf, [None, 1, None, 1, 1, 1, 1, 1]), (-75.0, [0, 1, None, math.exp(-1e33 * math.exp(-75.0)), 0, 1, 1, 1]), (inf, [0, None, None, 0, 0, 0, 0, 0])):
        y = H.matmul_nt(zero, eye, b, decay=torch.full((4,), act, device=DEV)).view(T, 16, 8)
        for i, v in enumerate(want):
            got = y[:, :, i]
            assert got.isnan().all() if v is None else ((got - v).abs() <= 1e-5 * v).all(), (act, i, got[0, 0])


# fp32 on 64 x 64 tiles of three blocks a CU: long plain and gated products of more than a round, rows and columns past the last tile's end, an odd number
# of K tiles, and row groups, empty and of one row among them, as they are and gathered; sums of 608 products in fp32: 1e-5 as above
@pytest.mark.parametrize("M,N", [(1100, 2056), (1037, 2056), (641, 4104)])
def test_three_blocks_a_unit(ops, M, N):
    H, _ = ops
    K = 608
    assert [H.k.fls_seq_gemm_tile_of(0, 0, M, N, K, 1, 0, g) for g in (0, 1)] == [6, 6]
    torch.manual_seed(M + N)
    a, w = torch.randn(M, K, device=DEV), 0.1 * torch.randn(N, K, device=DEV)
    z = a.double() @ w.double().t()
    close(H.matmul_nt(a, w), z, 1e-5)
    close(H.gated_matmul_nt(a, w, torch.float32), torch.nn.functional.silu(z[:, :N // 2]) * z[:, N // 2:], 2e-5)
    sizes, N = [0, M // 2, 1, M - M // 2 - 4, 0, 3], 6152
    assert [H.k.fls_seq_gemm_tile_of(0, 0, M, N, K, 6, 1, g) for g in (0, 1)] == ([6, 6] if M > 700 else [2, 2])
    offs, w = torch.tensor(np.cumsum([0] + sizes), dtype=torch.int32, device=DEV), 0.1 * torch.randn(6, N, K, device=DEV)
    y = lambda x: torch.cat([x[offs[e]:offs[e + 1]].double() @ w[e].double().t() for e in range(6)])
    close(H.grouped_matmul_nt(a, w, offs), y(a), 1e-5)
    rows = torch.randperm(M, device=DEV).to(torch.int32) // 2
    z = y(a[rows.long()])
    close(H.gated_matmul_nt(a[:(M + 1) // 2], w, torch.float32, offs=offs, rows=rows), torch.nn.functional.silu(z[:, :N // 2]) * z[:, N // 2:], 2e-5)


# few rows at the edges of what a pass takes; K of one lane's share, less than a K tile, a tile and a tail, more tiles than the waves' rings hold; columns
# past a block's end, one and several rounds of blocks.  Rows of infinities and NaN leave the others alone.  fp32 sums of up to 4,168 products: 1e-5 as above
@pytest.mark.parametrize("types", ["bf16", "mixed", "fp32"])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 24, 25, 32])
def test_few_rows_edges(ops, types, M):
    H, _ = ops
    ta, tw = {"bf16": (torch.bfloat16, torch.bfloat16), "mixed": (torch.float32, torch.bfloat16), "fp32": (torch.float32, torch.float32)}[types]
    f64 = lambda t: (t.to(tw) if types == "mixed" else t).double()
    torch.manual_seed(M)
    for N, K in ((20, 8), (268, 72), (4124, 200), (6440, 1032), (136, 4168)):
        a, w = torch.randn(M, K, device=DEV).to(ta), (0.1 * torch.randn(N, K, device=DEV)).to(tw)
        z = f64(a) @ w.double().t()
        close(H.matmul_nt(a, w), z, 1e-5)
        close(H.gated_matmul_nt(a, w, torch.float32), torch.nn.functional.silu(z[:, :N // 2]) * z[:, N // 2:], 2e-5)
        if M > 1:
            b = a.clone()
            b[M - 1, K // 2], b[M // 2 - 1, K - 1] = float("inf"), float("nan")
            y, rest = H.matmul_nt(b, w), [r for r in range(M) if r not in (M - 1, M // 2 - 1)]
            assert torch.equal(y[rest], H.matmul_nt(a, w)[rest]) and not y[[M - 1, M // 2 - 1]].isfinite().any()


# short rows about the lengths (256, 512 and 1024 bytes of a weight row, by rows, columns and gates) up to which operands go straight to registers: whole
# steps and tails, waves without a step, columns past a block's end, up to a round of blocks and more; row groups, empty and of more rows than a pass
# takes, as they are and gathered.  fp32 sums of up to 520 products: 1e-5 as above
@pytest.mark.parametrize("types", ["bf16", "mixed", "fp32"])
@pytest.mark.parametrize("terms", [128, 136, 248, 256, 264, 504, 512, 520])
def test_few_rows_of_few_terms(ops, types, terms):
    H, _ = ops
    ta, tw = {"bf16": (torch.bfloat16, torch.bfloat16), "mixed": (torch.float32, torch.bfloat16), "fp32": (torch.float32, torch.float32)}[types]
    f64 = lambda t: (t.to(tw) if types == "mixed" else t).double()
    gate = lambda z: torch.nn.functional.silu(z[:, :z.shape[1] // 2]) * z[:, z.shape[1] // 2:]
    K = terms // 2 // 8 * 8 if types == "fp32" else terms
    torch.manual_seed(terms)
    for M, N in ((1, 20), (16, 4096), (16, 4136), (5, 8200), (17, 4096), (32, 4104), (20, 8200)):
        a, w = torch.randn(M, K, device=DEV).to(ta), (0.1 * torch.randn(N, K, device=DEV)).to(tw)
        z = f64(a) @ w.double().t()
        close(H.matmul_nt(a, w), z, 1e-5)
        close(H.gated_matmul_nt(a, w, torch.float32), gate(z), 2e-5)
    sizes, N = [0, 1, 19, 0, 3, 0, 0, 2, 8], 136
    M = sum(sizes)
    offs, w = torch.tensor(np.cumsum([0] + sizes), dtype=torch.int32, device=DEV), (0.1 * torch.randn(len(sizes), N, K, device=DEV)).to(tw)
    a, rows = torch.randn(M, K, device=DEV).to(ta), torch.randperm(M, device=DEV).to(torch.int32)
    y = lambda x: torch.cat([f64(x[offs[e]:offs[e + 1]]) @ w[e].double().t() for e in range(len(sizes))])
    close(H.grouped_matmul_nt(a, w, offs), y(a), 1e-5)
    close(H.gated_matmul_nt(a, w, torch.float32, offs=offs), gate(y(a)), 2e-5)
    close(H.gated_matmul_nt(a, w, torch.float32, offs=offs, rows=rows), gate(y(a[rows.long()])), 2e-5)


# about the rows up to which row groups take the few-row kernel, spread over the groups and nearly all in one
@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("M", [64, 65, 128, 129])
def test_grouped_rows_in_one_group(ops, cdt, tol, M):
    H, R = ops
    torch.manual_seed(M)
    E, N, K = 20, 72, 192
    a, w = torch.randn(M, K, device=DEV).to(cdt), torch.randn(E, N, K, device=DEV).to(cdt)
    for sizes in ([M // E] * (E - 1) + [M - M // E * (E - 1)], [0, 1] + [0] * (E - 4) + [M - 2, 1]):
        offs = torch.tensor(np.cumsum([0] + sizes), dtype=torch.int32, device=DEV)
        close(H.grouped_matmul_nt(a, w, offs), R.grouped_matmul_nt(a, w, offs), 1e-5)


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_rows(ops, cdt, tol):
    H, R = ops
    torch.manual_seed(1)
    x = torch.randn(37, 96, device=DEV)
    w = torch.randn(96, device=DEV)
    idx = torch.tensor([3, 0, 36, 5], dtype=torch.int32, device=DEV)
    close(H.group_rmsnorm(x, w, 3, 1e-6, cdt), R.group_rmsnorm(x, w, 3, 1e-6, cdt), tol)
    close(H.group_rmsnorm(x, w, 1, 1e-6, cdt, row_idx=idx), R.group_rmsnorm(x, w, 1, 1e-6, cdt, row_idx=idx), tol)
    x1, x2, y = x.clone(), x.clone(), torch.randn(37, 96, device=DEV)
    close(H.add_group_rmsnorm_(x1, y, w, 2, 1e-6), R.add_group_rmsnorm_(x2, y, w, 2, 1e-6), 1e-5)
    u = torch.randn(9, 48, device=DEV)
    wg = torch.randn(6, 16, 16, device=DEV).to(cdt)
    bg = torch.randn(96, device=DEV)
    close(H.block_linear(u, wg, bg, 3, cdt), R.block_linear(u, wg, bg, 3, cdt), 1e-5)
    z = torch.randn(11, 50, device=DEV) * 3
    act = torch.tensor([0.3, -0.2], device=DEV)
    close(H.xielu(z, act, cdt), R.xielu(z, act, cdt), tol)
    close(H.silu_mul(z, cdt), R.silu_mul(z, cdt), tol)
    eye = torch.eye(50, device=DEV)
    close(H.matmul_nt(z, eye, softcap=5.0), R.matmul_nt(z, eye, softcap=5.0), 1e-5)
    assert bool((H.argmax_f32(z).cpu() == R.argmax_f32(z).cpu()).all())
    tab = torch.randn(40, 24, device=DEV).to(cdt)
    ids = torch.tensor([1, 39, 0, 7], dtype=torch.int32, device=DEV)
    close(H.embed_rows(ids, tab), R.embed_rows(ids, tab), 1e-6)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv", [(6, 2, 24, 40), (6, 2, 64, 64), (4, 4, 128, 64), (8, 2, 128, 128), (2, 1, 64, 128)])
def test_attention(ops, cdt, tol, Hh, G, d, dv):
    H, R = ops
    torch.manual_seed(d + dv)
    for lens, pos0, chunk, window in (([70, 5, 33], [0, 0, 0], 20, 0), ([3, 1, 1], [70, 5, 33], 20, 0), ([40, 17], [0, 0], 0, 9),
                                      ([2, 2], [40, 17], 0, 9), ([150], [0], 64, 0), ([300, 17, 140], [0, 0, 0], 100, 0),
                                      ([200, 30], [300, 17], 100, 0), ([260], [0], 0, 50), ([260], [0], 0, 0)):
        md, npages, _ = meta_of(lens, pos0, DEV)
        T = sum(lens)
        kc = torch.randn(npages, 16, G * d, device=DEV).to(cdt)
        vc = torch.randn(npages, 16, G * dv, device=DEV).to(cdt)
        kc2, vc2 = kc.clone(), vc.clone()
        k, v, kn = torch.randn(T, G * d, device=DEV), torch.randn(T, G * dv, device=DEV), torch.randn(G * d, device=DEV)
        H.kv_store(k, kn, 1e-6, v, kc, vc, md["kv_slot"])
        R.kv_store(k, kn, 1e-6, v, kc2, vc2, md["kv_slot"])
        close(kc, kc2, tol)
        close(vc, vc2, tol)
        q = torch.randn(T, Hh * d, device=DEV).to(cdt)
        r1, r2 = torch.rand(Hh, device=DEV), torch.rand(Hh, device=DEV)
        o1 = H.attn_paged(q, kc2, vc2, md, Hh, G, d, dv, 0.3, 8.0, r1, r2, chunk, 16, cdt, window=window)
        o2 = R.attn_paged(q, kc2, vc2, md, Hh, G, d, dv, 0.3, 8.0, r1, r2, chunk, 16, cdt, window=window)
        close(o1, o2, tol)


# values by four columns a lane (heads of 32, 64, 128 and 256) and by one (any other, or rows that vectors do not fit): keys about what a wave has
# side by side, has in flight, and about its tiles of 64, with windows, kept first keys and a second range.  fp32 pools against fp64: sums of up to
# 700 terms of either sign in fp32, 2e-5 of the largest
@pytest.mark.parametrize("dv", [32, 64, 128, 256, 36])
@pytest.mark.parametrize("d,pad", [(32, 0), (36, 0), (96, 0), (96, 2), (160, 4)])
def test_attention_values_by_columns(ops, dv, d, pad):
    H, _ = ops
    Hh, G = 4, 2
    pos0 = [0, 1, 6, 7, 8, 9, 14, 15, 16, 31, 32, 62, 63, 64, 65, 127, 128, 129, 255, 700]
    md, npages, _ = meta_of([1] * len(pos0), pos0, DEV)
    torch.manual_seed(dv + d)
    kc, vc = torch.randn(npages, 16, G * d, device=DEV), torch.randn(npages, 16, G * dv + pad, device=DEV)
    q = torch.randn(len(pos0), Hh * d, device=DEV)
    table, k64, v64 = md["page_table"].cpu().long(), kc.cpu().double().view(-1, G, d), vc.cpu().double().view(-1, G * dv + pad)[:, :G * dv]
    q64 = q.cpu().double().view(-1, Hh, d)
    for window, keep in ((0, 0), (20, 0), (70, 5)):
        got = H.attn_paged(q, kc, vc, md, Hh, G, d, dv, d ** -0.5, 0.0, None, None, 0, 16, torch.float32, window=window, keep_first=keep).cpu().double()
        for t, i in enumerate(pos0):
            lo = max(0, i - window + 1) if window else 0
            j = torch.tensor(list(range(min(keep, lo))) + list(range(lo, i + 1)))
            rows = table[t][j // 16] * 16 + j % 16
            kk, vv = k64[rows].repeat_interleave(Hh // G, 1), v64[rows].view(-1, G, dv).repeat_interleave(Hh // G, 1)
            p = torch.softmax(torch.einsum("hd,nhd->hn", q64[t], kk) * d ** -0.5, -1)
            want = torch.einsum("hn,nhv->hv", p, vv).reshape(-1)
            assert float((got[t] - want).abs().max()) < 2e-5 * float(want.abs().max()), (i, window)


# few rows on sixteen waves (256 rows x heads, ranges of keys among them) and the same rows too often for it on four: lengths about a tile of 16, a
# wave's turn of 256 and ranges of their own, every option, shared values, heads whose pieces do not divide by four lanes.  fp32 throughout, sums
# of up to 1,500 terms and weights of up to 20 in the exponent: 3e-5 of the largest
@pytest.mark.parametrize("d,dv", [(64, 32), (96, 64), (72, 128), (128, 256), (200, 128)])
@pytest.mark.parametrize("kind", ["plain", "penalty", "sigmoid", "sink"])
def test_attention_few_rows(ops, d, dv, kind):
    H, R = ops
    Hh, G = 4, 2
    torch.manual_seed(d + dv)
    r1, r2 = (torch.rand(Hh, device=DEV), torch.rand(Hh, device=DEV)) if kind == "penalty" else (None, None)
    kw = dict(gate_bias=torch.randn(Hh, device=DEV) - 2) if kind == "sigmoid" else \
        dict(sink=torch.randn(Hh, device=DEV), head_gate=torch.randn(100, Hh, device=DEV)) if kind == "sink" else {}
    for pos0, ps in (([0, 1, 14, 15, 16, 17, 63, 64, 240, 254, 255, 256, 257], 24), ([511, 512, 1500], 16)):
        md, npages, _ = meta_of([1] * len(pos0), pos0, DEV, ps)
        kc, vc = torch.randn(npages, ps, G * d, device=DEV), torch.randn(npages, ps, G * dv, device=DEV)
        q = torch.randn(len(pos0), Hh * d, device=DEV)
        for chunk, window, keep in ((0, 0, 0), (200, 0, 0), (0, 40, 0), (0, 40, 30)):
            for rep in (1, 100 // len(pos0)):
                m2 = dict(md, tok_seq=md["tok_seq"].repeat(rep), tok_pos=md["tok_pos"].repeat(rep))
                k2 = dict(kw, head_gate=kw["head_gate"][:rep * len(pos0)]) if "head_gate" in kw else kw
                args = (q.repeat(rep, 1), kc, vc, m2, Hh, G, d, dv, d ** -0.5, 20.0 if kind == "penalty" else 0.0, r1, r2, chunk, ps, torch.float32)
                o1, o2 = (o.attn_paged(*args, window=window, keep_first=keep, v_heads=1 if kind == "sigmoid" and dv < 256 else None, **k2) for o in (H, R))
                close(o1, o2, 3e-5)


# prompt attention over 64-key tiles in two halves: lengths about a half, a tile and a 128-row block, windows and chunks that end inside
# a half, kept first keys, pages of 24 (no power of two); `grow`: scores that rise along the keys in small steps or in large ones
# (the running maximum grows key by key, or in jumps), with a sink far below, near and far above them.  bf16 tolerance as above
@pytest.mark.parametrize("lens,pos0", [([31, 33], [0, 0]), ([64, 65], [0, 7]), ([129], [0]), ([200], [333])])
@pytest.mark.parametrize("d,dv,ps", [(64, 128, 24), (128, 128, 16)])
def test_prompt_attention_tiles(ops, lens, pos0, d, dv, ps):
    H, R = ops
    Hh, G, T = 4, 2, sum(lens)
    torch.manual_seed(T + d)
    md, npages, _ = meta_of(lens, pos0, DEV, ps)
    kc, vc = torch.randn(npages, ps, G * d, device=DEV).bfloat16(), torch.randn(npages, ps, G * dv, device=DEV).bfloat16()
    q = torch.randn(T, Hh * d, device=DEV).bfloat16()
    for chunk, window, keep in ((0, 0, 0), (45, 0, 0), (0, 37, 0), (0, 37, 5), (0, 100, 70)):
        for qq in (q, q.float()):
            o1, o2 = (o.attn_paged(qq, kc, vc, md, Hh, G, d, dv, d ** -0.5, 0.0, None, None, chunk, ps, torch.bfloat16, window=window,
                                   keep_first=keep) for o in (H, R))
            close(o1, o2, 2e-2)
    for step in (0.02, 0.9):
        order = torch.arange(max(p + n for p, n in zip(pos0, lens)), device=DEV, dtype=torch.float32)
        kg = kc.clone().view(npages * ps, G, d)
        for b in range(len(lens)):
            j = torch.arange(pos0[b] + lens[b], device=DEV)
            rows = md["page_table"][b].long()[j // ps] * ps + j % ps
            kg[rows, :, 0] = (order[:len(j), None] * step).bfloat16()
        qg = q.clone().view(T, Hh, d)
        qg[:, :, 0] = 1.0
        for sink in (None, -20.0, 5.0, 60.0):
            kw = {} if sink is None else dict(sink=sink)
            o1, o2 = (o.attn_paged(qg.view(T, -1), kg.view(npages, ps, G * d), vc, md, Hh, G, d, dv, 0.3, 0.0, None, None, 0, ps,
                                   torch.bfloat16, **kw) for o in (H, R))
            close(o1, o2, 2e-2)


# a query's largest weight is exactly 1 whatever came before it: every other key's value is 0, so the output is that key's value over the sum of
# weights to fp32, at jumps of 0.1 to 6 over the keys before and with a sink and the cap (two bf16 terms of any other weight: 7.6e-6)
@pytest.mark.parametrize("d,dv", [(64, 128), (128, 64)])
@pytest.mark.parametrize("cap,sink", [(0.0, None), (0.0, 0.05), (30.0, None)])
def test_prompt_attention_largest_weight(ops, d, dv, cap, sink):
    H, _ = ops
    Hh, n, at = 16, 100, 70
    md, npages, _ = meta_of([n], [0], DEV)
    jump = torch.linspace(0.1, 6.0, Hh).bfloat16()
    q, k, v = torch.zeros(n, Hh, d), torch.zeros(n, d), torch.zeros(n, dv)
    q[:, :, 0], k[at, 0], v[at] = jump.float(), 1.0, torch.randn(dv, generator=torch.Generator().manual_seed(d)).bfloat16().float()
    kc, vc = torch.zeros(npages, 16, d).bfloat16(), torch.zeros(npages, 16, dv).bfloat16()
    tab, j = md["page_table"][0].cpu().long(), torch.arange(n)
    kc.view(-1, d)[tab[j // 16] * 16 + j % 16], vc.view(-1, dv)[tab[j // 16] * 16 + j % 16] = k.bfloat16(), v.bfloat16()
    out = torch.empty(n, Hh * dv, device=DEV)
    H.attn_paged(q.bfloat16().view(n, -1).to(DEV), kc.to(DEV), vc.to(DEV), md, Hh, 1, d, dv, 1.0, cap, None, None, 0, 16, torch.bfloat16, out=out,
                 **({} if sink is None else dict(sink=sink)))
    s = jump.double()
    s = cap * torch.tanh(s / cap) if cap else s
    for i in range(at, n):
        w = torch.exp(s) / (torch.exp(s) + i + (0.0 if sink is None else math.exp(sink)))
        want = w[:, None] * v[at].double()
        assert float(((out[i].cpu().double().view(Hh, dv) - want).abs() / want.abs().clamp(min=1e-30)).max()) < 1e-6
    assert not bool(out[:at].any())


# every kind of weight (softmax, cap, penalty, both, sigmoid) with heads that go to the XCDs by groups (8, 16) and as they come (6), lengths
# about a half, a tile and a block, pages no tile fits, carried positions.  fp32 results: weights of two bf16 terms (2^-17), scores of up to
# 30 in units of log 2 to fp32 (2e-6 each side, and 2e-6 for exp's own): 3e-5
@pytest.mark.parametrize("Hh,G", [(8, 2), (16, 16), (6, 3)])
@pytest.mark.parametrize("lens,pos0", [([32, 1, 63], [0, 300, 1]), ([128, 33], [0, 95]), ([257], [64])])
@pytest.mark.parametrize("kind", ["plain", "cap", "penalty", "both", "sigmoid"])
def test_prompt_attention_kinds(ops, Hh, G, lens, pos0, kind):
    H, R = ops
    T, d, ps = sum(lens), 128, 24
    torch.manual_seed(T + Hh)
    md, npages, _ = meta_of(lens, pos0, DEV, ps)
    kc, vc = torch.randn(npages, ps, G * d, device=DEV).bfloat16(), torch.randn(npages, ps, G * d, device=DEV).bfloat16()
    q = torch.randn(T, Hh * d, device=DEV).bfloat16()
    r1, r2 = (torch.rand(Hh, device=DEV), torch.rand(Hh, device=DEV)) if kind in ("penalty", "both") else (None, None)
    cap = 8.0 if kind in ("cap", "both") else 0.0
    kw = dict(gate_bias=torch.randn(Hh, device=DEV) - 2) if kind == "sigmoid" else {}
    for chunk, window, keep in ((0, 0, 0), (100, 0, 0), (0, 70, 0), (0, 70, 40)):
        o1, o2 = torch.empty(T, Hh * d, device=DEV), torch.empty(T, Hh * d, device=DEV)
        for o, out in ((H, o1), (R, o2)):
            o.attn_paged(q, kc, vc, md, Hh, G, d, d, d ** -0.5, cap, r1, r2, chunk, ps, torch.bfloat16, window=window, keep_first=keep, out=out, **kw)
        close(o1, o2, 3e-5)


# every distance's penalty at its place: queries of zeros, so that a weight is (1 + r2 distance)^-r1 alone, and values that are the key's
# unit vector, so that each output is one weight.  Two bf16 terms of a weight (2^-17) and fp32 logarithms of up to 10 times r1 <= 3: 3e-5
# of the weight; none for a key behind the query
@pytest.mark.parametrize("n,pos0", [(128, 0), (97, 31), (33, 95), (32, 64), (70, 1)])
@pytest.mark.parametrize("sigmoid", [False, True])
def test_prompt_attention_penalty_of_every_distance(ops, n, pos0, sigmoid):
    H, _ = ops
    Hh, G, d, keys = 8, 2, 128, pos0 + n
    md, npages, _ = meta_of([n], [pos0], DEV)
    kc, vc = torch.randn(npages, 16, G * d, device=DEV).bfloat16(), torch.zeros(npages, 16, G, d, device=DEV).bfloat16()
    j = torch.arange(keys, device=DEV)
    vc.view(-1, G, d)[md["page_table"][0].long()[j // 16] * 16 + j % 16, :, j] = 1.0
    r1, r2 = torch.linspace(0.1, 3.0, Hh, device=DEV), torch.linspace(2.0, 0.01, Hh, device=DEV)
    bias = torch.linspace(-2, 1, Hh, device=DEV)
    out = torch.empty(n, Hh * d, device=DEV)
    H.attn_paged(torch.zeros(n, Hh * d, device=DEV).bfloat16(), kc, vc.view(npages, 16, G * d), md, Hh, G, d, d, 0.1, 0.0, r1, r2, 0, 16,
                 torch.bfloat16, out=out, **(dict(gate_bias=bias) if sigmoid else {}))
    dist = (torch.arange(pos0, keys)[:, None] - torch.arange(keys)[None, :]).double()
    s = -r1.cpu().double()[:, None, None] * torch.log1p(r2.cpu().double()[:, None, None] * dist.clamp(min=0))
    s = torch.where(dist >= 0, s, -torch.inf)
    want = torch.sigmoid(s + bias.cpu().double()[:, None, None]) if sigmoid else torch.softmax(s, -1)
    got = out.cpu().double().view(n, Hh, d)[:, :, :keys].permute(1, 0, 2)
    assert bool(((got - want).abs() <= 3e-5 * want).all())
    assert not bool(out.view(n, Hh, d)[:, :, keys:].any())


# norms with rows in registers: one to eight steps of 1024 columns a group, the last one partly filled, the widest and the first beyond it
# (8192, 8196), odd widths and strides that go to the general kernel, one weight for all columns; the residual update with the
# next norm against the two in turn.  fp32 outputs against fp64: sums of up to 8196 squares in a tree, 1e-6; bf16 rounding 2^-8
@pytest.mark.parametrize("n,groups", [(4, 3), (1020, 1), (1024, 2), (1028, 2), (2052, 1), (4096, 1), (4100, 2), (8192, 1), (8196, 1), (30, 2)])
def test_norm_widths(ops, n, groups):
    H, _ = ops
    torch.manual_seed(n)
    D = n * groups
    norm = lambda x, w: (x.reshape(-1, groups, n) / (x.reshape(-1, groups, n).pow(2).mean(-1, keepdim=True) + 1e-6).sqrt()).reshape(-1, D) * w
    w, w2 = torch.randn(D, device=DEV), torch.randn(D, device=DEV)
    for pad in (0, 4, 3):
        x, y = (torch.randn(5, D + pad, device=DEV)[:, :D] for _ in range(2))
        x6, y6, w6, v6 = (t.cpu().double() for t in (x, y, w, w2))
        close(H.group_rmsnorm(x, w, groups, 1e-6, torch.float32, w_offset=1.0), norm(x6, w6 + 1), 1e-6)
        close(H.group_rmsnorm(x, w, groups, 1e-6, torch.bfloat16), norm(x6, w6), 2 ** -8)
        close(H.group_rmsnorm(x, w[:1], groups, 1e-6, torch.float32), norm(x6, w6[:1]), 1e-6)
        for cdt, tol in ((torch.float32, 1e-6), (torch.bfloat16, 2 ** -8)):
            x1 = torch.empty(5, D + pad, device=DEV)[:, :D].copy_(x)
            h = H.add_group_rmsnorm_next_(x1, y, w, w2, groups, 1e-6, cdt)
            new = x6 + norm(y6, w6)
            close(x1, new, 1e-6)
            close(h, norm(new, v6), tol)


# the residual update of a mixture: rows summed on the way into the norm, one to many choices, widths as above and one for the general
# kernels, tokens on both sides of the one-launch routing; fp32 sums in the oracle's order
@pytest.mark.parametrize("T", [3, 70])
@pytest.mark.parametrize("D,groups,E,top", [(24, 3, 5, 1), (2048, 2, 20, 4), (4100, 1, 40, 16), (30, 2, 6, 3)])
def test_mixture_into_norm(ops, T, D, groups, E, top):
    H, R = ops
    torch.manual_seed(D + T)
    route = H.moe_route_corrected(torch.randn(T, E, device=DEV), torch.randn(E, device=DEV) * 0.1, top)
    y, w, x = torch.randn(T * top, D, device=DEV), torch.randn(D, device=DEV), torch.randn(T, D, device=DEV)
    y6 = (y.cpu().double()[route.dest.cpu().long()] * route.w.cpu().double()[:, :, None]).sum(1).reshape(T, groups, -1)
    want = x.cpu().double() + (y6 / (y6.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt()).reshape(T, D) * w.cpu().double()
    close(H.add_group_rmsnorm_moe_(x, y, route, w, groups, 1e-6), want, 1e-6)


# activations with bf16 results from the tiles' epilogues, element by element over the bf16 range (tiny, about the forms' seam at -1/2, large,
# infinite): within a rounding of the fp64 value (2^-8 relative; a sigmoid
# below 2^-126 may be flushed, and a result)
@pytest.mark.parametrize("kind", ["xielu", "silu", "gelu_tanh", "clamped"])
def test_epilogue_bf16_values(ops, kind):
    H, _ = ops
    g = torch.Generator().manual_seed(5)
    z = torch.cat([torch.linspace(-1, 1, 300), torch.logspace(-30, 2, 300, base=2.0) * torch.where(torch.rand(300, generator=g) < 0.5, -1.0, 1.0),
                   torch.linspace(-90, 90, 150), torch.tensor([0.0, -0.0, -0.5, 0.5, 3e4, -3e4])]).bfloat16()
    M, N, K = z.numel(), 256, 64
    a = torch.zeros(M, K, dtype=torch.bfloat16)
    a[:, 0], a[:, 1] = z, z.flip(0)
    z6, u6 = z.double(), z.flip(0).double()
    if kind == "xielu":
        act = torch.tensor([0.3, -0.2])
        w = torch.zeros(N, K)
        w[:, 0] = 1
        got = H.matmul_nt(a.to(DEV), w.bfloat16().to(DEV), xielu=act.to(DEV), out_dtype=torch.bfloat16)
        p, q = torch.nn.functional.softplus(act.double())
        want = torch.where(z6 > 0, p * z6 * z6, (0.5 + q) * (torch.expm1(z6) - z6)) + 0.5 * z6
    else:
        w = torch.zeros(2 * N, K)
        w[:N, 0], w[N:, 1] = 1, 1
        got = H.gated_matmul_nt(a.to(DEV), w.bfloat16().to(DEV), torch.bfloat16, act=kind, limit=7.0, alpha=1.702)
        if kind == "silu":
            want = z6 * torch.sigmoid(z6) * u6
        elif kind == "gelu_tanh":
            want = z6 * torch.sigmoid(2 * (2 / torch.pi) ** 0.5 * (z6 + 0.044715 * z6 ** 3)) * u6
        else:
            zc = z6.clamp(max=7.0)
            want = zc * torch.sigmoid(1.702 * zc) * (u6.clamp(-7.0, 7.0) + 1)
    err = (got.cpu().double() - want[:, None]).abs()
    assert bool((err <= want[:, None].abs() * 2 ** -8 + (1 + (z6 * (u6.abs() + 1)).abs())[:, None] * 2.0 ** -126).all())


# results that go to pinned host memory by the kernels that make them: the few-row product's rows bit for bit (32 rows are its most, blocks of 32
# columns from 6,400 on), or, where another kernel takes the product (more rows, columns that are no multiple of 4), the rows by the
# argmax; the argmax behind them; a cell of 0: nowhere
@pytest.mark.parametrize("M", [1, 3, 16, 17, 32, 33])
@pytest.mark.parametrize("N", [4, 20, 1000, 4100, 6400, 6404, 510, 1023])
@pytest.mark.parametrize("cdt", [torch.bfloat16, torch.float32])
def test_rows_written_to_the_host(ops, M, N, cdt):
    H, _ = ops
    g = torch.Generator().manual_seed(M + N)
    a, w = torch.randn(M, 256, generator=g).to(cdt).to(DEV), torch.randn(N, 256, generator=g).to(cdt).to(DEV)
    down = torch.full((M * N + M + 4,), -7.0, pin_memory=True)
    cell = torch.tensor([down.data_ptr()], dtype=torch.int64, device=DEV)
    for how in ({}, dict(softcap=5.0)):
        down.fill_(-7.0)
        mirror = H.host_rows(cell)
        c = H.matmul_nt(a, w, mirror=mirror, **how)
        assert mirror.rows_there == (M <= 32 and N % 4 == 0)
        am = H.argmax_f32(c, mirror)
        torch.cuda.synchronize()
        assert torch.equal(c, H.matmul_nt(a, w, **how)) and torch.equal(am.cpu().long(), c.argmax(1).cpu())
        assert torch.equal(down[:M * N].view(M, N), c.cpu()) and torch.equal(down[M * N:M * N + M].view(torch.int32), am.cpu())
        assert bool((down[M * N + M:] == -7.0).all())
        down.fill_(-7.0)
        nowhere = H.host_rows(torch.zeros(1, dtype=torch.int64, device=DEV))
        assert torch.equal(c, H.matmul_nt(a, w, mirror=nowhere, **how)) and torch.equal(am, H.argmax_f32(c, nowhere))
        torch.cuda.synchronize()
        assert bool((down == -7.0).all())


# the same for rows long enough for the rings, blocks of 16 and of 32 columns
@pytest.mark.parametrize("M,N", [(1, 4), (8, 1000), (16, 6404), (17, 4100), (32, 6404), (9, 16400)])
@pytest.mark.parametrize("cdt", [torch.bfloat16, torch.float32])
def test_long_rows_written_to_the_host(ops, M, N, cdt):
    H, _ = ops
    torch.manual_seed(M + N)
    a, w = torch.randn(M, 1032, device=DEV).to(cdt), torch.randn(N, 1032, device=DEV).to(cdt)
    down = torch.full((M * N + 4,), -7.0, pin_memory=True)
    mirror = H.host_rows(torch.tensor([down.data_ptr()], dtype=torch.int64, device=DEV))
    c = H.matmul_nt(a, w, mirror=mirror)
    torch.cuda.synchronize()
    assert mirror.rows_there and torch.equal(c, H.matmul_nt(a, w))
    assert torch.equal(down[:M * N].view(M, N), c.cpu()) and bool((down[M * N:] == -7.0).all())


# weight rows so far apart (2^27 elements: past the few-row kernel's 32-bit offsets) that another kernel takes the product: the argmax then
# writes the rows
def test_rows_written_to_the_host_of_far_weight_rows(ops):
    H, _ = ops
    M, N, K = 3, 4, 64
    w = torch.empty_strided((N, K), (2 ** 27, 1), dtype=torch.bfloat16, device=DEV).copy_(torch.randn(N, K))
    a = torch.randn(M, K, device=DEV).bfloat16()
    down = torch.full((M * N + M,), -7.0, pin_memory=True)
    mirror = H.host_rows(torch.tensor([down.data_ptr()], dtype=torch.int64, device=DEV))
    c = H.matmul_nt(a, w, mirror=mirror)
    am = H.argmax_f32(c, mirror)
    torch.cuda.synchronize()
    close(c, a.float() @ w.float().t(), 1e-5)
    assert not mirror.rows_there
    assert torch.equal(down[:M * N].view(M, N), c.cpu()) and torch.equal(down[M * N:].view(torch.int32), am.cpu())


@pytest.mark.parametrize("n", [1, 3, 4, 64, 4095, 4096, 4097, 9001])
def test_copy_words_from_the_host(ops, n):
    H, _ = ops
    src = torch.randint(-2 ** 31, 2 ** 31 - 1, (n,), dtype=torch.int32).pin_memory()
    dst = torch.full((n + 8,), 5, dtype=torch.int32, device=DEV)
    H.copy_words(src, dst[:n])
    assert torch.equal(dst[:n].cpu(), src) and bool((dst[n:] == 5).all())


# xIELU's negative side on both sides of its seam at -1, near 0 (where exp(z) - 1 cancels) and far out, against fp64: 3 ulp of
# (exp(z) - 1 - z) (1/2 + softplus(q)) and one of each of the sums' terms
def test_xielu_against_fp64(ops):
    H, _ = ops
    act = torch.tensor([0.3, -0.2])
    p, q = torch.nn.functional.softplus(act.double())
    ap, an = p, 0.5 + q
    z = torch.cat([torch.linspace(a, b, 4096) for a, b in ((-100, -20), (-20, -1), (-1.01, -0.99), (-1, 0), (-1e-2, 0), (-1e-4, 0), (0, 5))]
                  + [torch.tensor([-1.0, -0.99999994, -1.0000001, -0.0, 0.0, -200.0, -1e30, 1e-30, -1e-30])])
    d = z.double()
    low = torch.where(d > -1e-2, d * d * (0.5 + d * (1 / 6 + d * (1 / 24 + d / 120))), torch.expm1(d) - d)
    want = torch.where(d > 0, ap * d * d, an * low) + 0.5 * d
    got = H.xielu(z[None].to(DEV), act.to(DEV), torch.float32).cpu().double()[0]
    ulp = 2.0 ** -23
    assert bool(((got - want).abs() <= ulp * (3 * torch.where(d > 0, ap * d * d, an * low) + 0.5 * d.abs() + want.abs()) + 1e-44).all())
    assert torch.isnan(H.xielu(torch.tensor([[float("nan")]], device=DEV), act.to(DEV), torch.float32)).all()


# an activation of the same sum has the same bits from the few-row kernel, the tiles and the kernels for any size (every sum here is one
# product, exact in any order)
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_epilogue_values_do_not_depend_on_the_rows(ops, out):
    H, _ = ops
    g = torch.Generator().manual_seed(6)
    M, N, K = 2080, 256, 64
    z, u = (3 * torch.randn(M, generator=g)).bfloat16(), torch.randn(N, generator=g).abs().bfloat16()
    a, w = torch.zeros(M, K, dtype=torch.bfloat16), torch.zeros(2 * N, K, dtype=torch.bfloat16)
    a[:, 0], a[:, 1], w[:N, 0], w[N:, 1] = z, z.flip(0), 1 + u / 8, u
    a, w, act = a.to(DEV), w.to(DEV), torch.tensor([0.3, -0.2], device=DEV)
    ragged = torch.zeros(M, K + 3, dtype=torch.bfloat16, device=DEV)[:, :K]
    ragged.copy_(a)
    for how in (dict(xielu=act), dict(relu2=True), dict(softcap=3.0), dict(scale=0.3), dict(decay=act)):
        f = lambda x: H.matmul_nt(x, w, out_dtype=out, **how)
        whole = f(a)
        assert torch.equal(whole, torch.cat([f(a[i:i + 32]) for i in range(0, M, 32)])) and torch.equal(whole, f(ragged)), how
    for kind in ("silu", "gelu_tanh", "clamped"):
        f = lambda x: H.gated_matmul_nt(x, w, out, act=kind, limit=7.0)
        whole = f(a)
        assert torch.equal(whole, torch.cat([f(a[i:i + 32]) for i in range(0, M, 32)])) and torch.equal(whole, f(ragged)), kind


# plain products of few columns that four-column stores don't fit: one column at a time from the tiles, rows about a tile's, all three
# operand types; sums of 256 products against fp64
@pytest.mark.parametrize("N", [1, 3, 10, 33, 62, 127])
@pytest.mark.parametrize("ta,tw,tol", [(torch.bfloat16, torch.bfloat16, 1e-6), (torch.float32, torch.bfloat16, 5e-3), (torch.float32, torch.float32, 1e-6)])
def test_matmul_few_columns(ops, N, ta, tw, tol):
    H, _ = ops
    torch.manual_seed(N)
    w = torch.randn(N, 256, device=DEV).to(tw)
    for M in (33, 64, 129, 1000):
        a = torch.randn(M, 256, device=DEV).to(ta)
        want = a.cpu().double() @ w.cpu().double().t()
        close(H.matmul_nt(a, w), want, tol)
        close(H.matmul_nt(a, w, out_dtype=torch.bfloat16), want, max(tol, 2 ** -8))


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_conv_and_scans_carry_state(ops, cdt, tol):
    H, R = ops
    torch.manual_seed(3)
    for lens, pos0 in (([9, 1, 4], [0, 0, 0]), ([2, 1, 1], [9, 1, 4]), ([1, 1, 1], [11, 2, 5]), ([40, 3], [0, 7]), ([300, 5, 129], [0, 0, 6])):
        md, _, nslots = meta_of(lens, pos0, DEV)
        T, C, taps = sum(lens), 70, 4
        x = torch.randn(T, C + 6, device=DEV)[:, 3:3 + C]
        w, b = torch.randn(C, taps, device=DEV), torch.randn(C, device=DEV)
        st = torch.randn(nslots, taps - 1, C, device=DEV)
        st2 = st.clone()
        close(H.causal_conv(x, w, b, st, md, "silu"), R.causal_conv(x, w, b, st2, md, "silu"), 1e-5)
        close(st, st2, 1e-6)
        Wd = 70
        u, g = torch.randn(T, Wd, device=DEV), torch.randn(T, 2 * Wd, device=DEV)
        lam, y = torch.randn(Wd, device=DEV), torch.randn(T, Wd, device=DEV)
        s1 = torch.randn(nslots, Wd, device=DEV)
        s2 = s1.clone()
        close(H.rglru_scan(u, g, lam, y, s1, md, 8.0, cdt), R.rglru_scan(u, g, lam, y, s2, md, 8.0, cdt), tol)
        close(s1, s2, 1e-5)
        for nh, P, N, Gg in ((6, 20, 24, 2), (4, 64, 128, 1), (3, 8, 16, 3), (2, 40, 200, 1)):
            inner = nh * P
            xbc = torch.randn(T, inner + 2 * Gg * N, device=DEV)
            zz, dt = torch.randn(T, inner, device=DEV), torch.randn(T, nh, device=DEV)
            dtb, Al, Ds = torch.randn(nh, device=DEV), torch.randn(nh, device=DEV) * 0.5, torch.randn(nh, device=DEV)
            s1 = torch.randn(nslots, nh, N, P, device=DEV)
            s2 = s1.clone()
            close(H.ssd_scan(xbc, zz, dt, dtb, Al, Ds, s1, md, nh, P, N, Gg), R.ssd_scan(xbc, zz, dt, dtb, Al, Ds, s2, md, nh, P, N, Gg), 3e-5)
            close(s1, s2, 3e-5)


# the chunked state-space scan: chunk ends, one row, a carried state, one and two column tiles a block, groups; the oracle in fp64 (a
# decay as strong as exp(-30) a row: differences of running sums must not lose it)
@pytest.mark.parametrize("lens,pos0,nh,P,N,G,strong", [((64, 1, 65), (0, 7, 0), 4, 16, 64, 2, 0.0), ((200,), (5,), 2, 48, 128, 1, 0.0),
                                                       ((24, 128), (0, 0), 2, 32, 128, 1, 3.0), ((40, 90), (0, 3), 128, 32, 64, 1, 0.0)])
def test_ssd_chunks(ops, lens, pos0, nh, P, N, G, strong):
    H, R = ops
    torch.manual_seed(sum(lens))
    md, _, nslots = meta_of(lens, pos0, DEV)
    T, inner = sum(lens), nh * P
    xbc = torch.randn(T, inner + 2 * G * N, device=DEV)
    z, dt = torch.randn(T, inner, device=DEV), torch.randn(T, nh, device=DEV)
    dtb, Al, Ds = torch.randn(nh, device=DEV), torch.randn(nh, device=DEV) * 0.5 + strong, torch.randn(nh, device=DEV)
    s1 = torch.randn(nslots, nh, N, P, device=DEV)
    s2 = s1.cpu().double()
    got = H.ssd_scan(xbc, z, dt, dtb, Al, Ds, s1, md, nh, P, N, G)
    x, B, C = (t.cpu().double() for t in torch.split(xbc, [inner, G * N, G * N], 1))
    dtv = torch.nn.functional.softplus((dt + dtb).cpu().double())
    dec = torch.exp(-torch.exp(Al.cpu().double()) * dtv)
    want = torch.empty(T, inner, dtype=torch.float64)
    for s, (n, p0) in enumerate(zip(lens, pos0)):
        a0, slot = int(md["cu_host"][s]), int(md["slot"][s])
        S = s2[slot] if p0 else torch.zeros(nh, N, P, dtype=torch.float64)
        for t in range(a0, a0 + n):
            Bt, Ct = (v[t].reshape(G, N).repeat_interleave(nh // G, 0) for v in (B, C))
            S = dec[t][:, None, None] * S + dtv[t][:, None, None] * Bt[:, :, None] * x[t].reshape(nh, 1, P)
            want[t] = ((S * Ct[:, :, None]).sum(1) + Ds.cpu().double()[:, None] * x[t].reshape(nh, P)).reshape(-1)
        s2[slot] = S
    close(got, want * torch.nn.functional.silu(z.cpu().double()), 3e-6)
    close(s1, s2, 3e-6)


# a step described without its longest request is walked row by row
def test_ssd_scan_without_the_longest_request(ops):
    H, R = ops
    torch.manual_seed(8)
    nh, P, N = 2, 16, 64
    md, _, nslots = meta_of([40, 3], [0, 5], DEV)
    args = [torch.randn(43, n, device=DEV) for n in (nh * P + 2 * N, nh * P, nh)] + [torch.randn(nh, device=DEV) for _ in range(3)]
    s1 = torch.randn(nslots, nh, N, P, device=DEV)
    s2 = s1.clone()
    got = H.ssd_scan(*args, s1, {k: v for k, v in md.items() if k != "max_rows"}, nh, P, N, 1)
    close(got, R.ssd_scan(*args, s2, md, nh, P, N, 1), 3e-5)
    close(s1, s2, 3e-5)


# a step so large that its own decay is 0 and the sum of a chunk's exponents would lose those of the rows after it
@pytest.mark.parametrize("step", [3e2, 1e12, 1e17, 1e25])
def test_ssd_chunks_huge_step(ops, step):
    H, _ = ops
    torch.manual_seed(7)
    n, P, N = 60, 16, 64
    md, _, nslots = meta_of((n,), (4,), DEV)
    xbc, z, dt = torch.randn(n, P + 2 * N, device=DEV), torch.randn(n, P, device=DEV), torch.randn(n, 1, device=DEV) - 2
    dt[20, 0] = step
    st, one = torch.randn(nslots, 1, N, P, device=DEV), torch.zeros(1, device=DEV)
    S, slot = st[int(md["slot"][0]), 0].cpu().double(), int(md["slot"][0])
    x, B, C = (t.cpu().double() for t in torch.split(xbc, [P, N, N], 1))
    d, want = torch.nn.functional.softplus(dt.cpu().double())[:, 0], torch.empty(n, P, dtype=torch.float64)
    for t in range(n):
        S = torch.exp(-d[t]) * S + d[t] * B[t][:, None] * x[t]
        want[t] = C[t] @ S
    got = H.ssd_scan(xbc, z, dt, one, one, one, st, md, 1, P, N, 1)
    want = want * torch.nn.functional.silu(z.cpu().double())
    close(got[:20], want[:20], 3e-6)
    close(got[20:], want[20:], 3e-6)
    close(st[slot, 0], S, 3e-6)


# the chunked scan is no further from 64 bits than the row-by-row kernel (both repeat themselves exactly; 3% for another card's sums).  Rates
# about exp(-1), steps about 0.4: a row decays by some 0.85; then by 0.5 and 0.98, at the first of which outputs are what is compared
@pytest.mark.parametrize("P,N", [(16, 64), (16, 128)])
@pytest.mark.parametrize("rate", [-1.0, 0.8, -4.0])
def test_ssd_chunks_are_as_exact_as_rows(ops, monkeypatch, P, N, rate):
    H, _ = ops
    torch.manual_seed(N)
    nh, lens = 64, (130, 300, 413, 500, 601)
    md, _, nslots = meta_of(lens, [0] * len(lens), DEV)
    T = sum(lens)
    xbc, z, dt = torch.randn(T, nh * P + 2 * N, device=DEV), torch.randn(T, nh * P, device=DEV), 0.5 * torch.randn(T, nh, device=DEV)
    dtb, Al, Ds = torch.randn(nh, device=DEV) - 1, 0.7 * torch.randn(nh, device=DEV) + rate, torch.randn(nh, device=DEV)
    x, B, C = (t.double() for t in torch.split(xbc, [nh * P, N, N], 1))
    d = torch.nn.functional.softplus((dt + dtb).double())
    e, o, states, t = torch.exp(-torch.exp(Al.double()) * d), torch.empty(T, nh, P, device=DEV).double(), [], 0
    for n in lens:
        S = torch.zeros(nh, N, P, device=DEV).double()
        for t in range(t, t + n):
            xt = x[t].reshape(nh, P)
            S = e[t][:, None, None] * S + d[t][:, None, None] * B[t][None, :, None] * xt[:, None, :]
            o[t] = (S * C[t][None, :, None]).sum(1) + Ds.double()[:, None] * xt
        states.append(S)
        t += 1
    want, err = (o.reshape(T, -1) * torch.nn.functional.silu(z.double()), torch.stack(states)), []
    for rows in (10 ** 9, 1):
        monkeypatch.setattr(H, "SSD_CHUNK_ROWS", rows)
        st = torch.zeros(nslots, nh, N, P, device=DEV)
        got = H.ssd_scan(xbc, z, dt, dtb, Al, Ds, st, md, nh, P, N, 1)
        err.append([float((a.double() - b).norm() / b.norm()) for a, b in zip((got, st[md["slot"].long()]), want)])
    assert err[1][0] <= 1.03 * err[0][0] and (rate > 0 or err[1][1] <= 1.03 * err[0][1]), err


# a value that is not finite stays where the recurrence puts it: rows before its own, other requests and (a value of x) other columns are
# what they are without it, bit by bit.  Rows in the first, a middle and the last block of 16 of a chunk, and in the second chunk
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("nh,P,N", [(2, 16, 64), (2, 48, 128), (128, 32, 128)])
def test_ssd_chunks_values_that_are_not_finite(ops, bad, nh, P, N):
    H, _ = ops
    torch.manual_seed(P + N)
    lens, pos0, inner = (100, 70), (0, 3), nh * P
    md, _, nslots = meta_of(lens, pos0, DEV)
    T, a1 = sum(lens), int(md["cu_host"][1])
    xbc, z, dt = torch.randn(T, inner + 2 * N, device=DEV), torch.randn(T, inner, device=DEV), torch.randn(T, nh, device=DEV)
    dtb, Al, Ds = torch.randn(nh, device=DEV), torch.randn(nh, device=DEV) * 0.5, torch.randn(nh, device=DEV)
    s0 = torch.randn(nslots, nh, N, P, device=DEV)
    other = int(md["slot"][1])

    def run(x, d):
        st = s0.clone()
        return H.ssd_scan(x, z, d, dtb, Al, Ds, st, md, nh, P, N, 1), st

    clean, sclean = run(xbc, dt)
    for t in (5, 44, 63, 90):
        for col in (3, inner + 2, inner + N + 2):                       # of x, B and C
            x = xbc.clone()
            x[t, col] = bad
            got, st = run(x, dt)
            assert torch.equal(got[:t], clean[:t]) and torch.equal(got[a1:], clean[a1:]) and torch.equal(st[other], sclean[other])
            assert not bool(got[t, :P].isfinite().all())
            if col == 3:
                keep = torch.arange(inner, device=DEV) != 3
                assert torch.equal(got[:, keep], clean[:, keep]) and not bool(got[t, 3].isfinite())
        d = dt.clone()
        d[t, 0] = bad
        got, st = run(xbc, d)                                           # (a step of -inf is one of size 0)
        assert torch.equal(got[:t], clean[:t]) and torch.equal(got[a1:], clean[a1:]) and torch.equal(st[other], sclean[other])
        assert torch.equal(got[:, P:], clean[:, P:]) and (bad < 0 or not bool(got[t, :P].isfinite().all()))


# the gated linear recurrence in one pass over the rows (32 channels a block, and 64 where the requests fill the chip) and in three over row
# tiles: parts and rounds of 128 rows that end early, one-row requests beside long ones, carried states; the oracle in fp64
@pytest.mark.parametrize("lens,W,limit", [([300, 1, 129, 16], 70, 10 ** 9), ([300, 1, 129, 16], 70, 0), ([1, 128, 3, 130] * 35, 130, 0)])
def test_rglru_forms(ops, monkeypatch, lens, W, limit):
    H, _ = ops
    torch.manual_seed(W)
    monkeypatch.setattr(H, "RGLRU_ROWS", limit)
    pos0 = [5 * (i % 2) for i in range(len(lens))]
    md, _, nslots = meta_of(lens, pos0, DEV)
    T = sum(lens)
    u, g, lam, y = torch.randn(T, W, device=DEV), torch.randn(T, 2 * W, device=DEV), torch.randn(W, device=DEV), torch.randn(T, W, device=DEV)
    st = torch.randn(nslots, W, device=DEV)
    want, out = st.cpu().double(), torch.empty(T, W, dtype=torch.float64)
    u6, g6, l6, y6 = (t.cpu().double() for t in (u, g, lam, y))
    la = -8.0 * torch.sigmoid(g6[:, :W]) * torch.nn.functional.softplus(l6)
    a6, b6 = torch.exp(la), torch.sqrt(-torch.expm1(2 * la)) * torch.sigmoid(g6[:, W:]) * u6
    for s, (n, p0) in enumerate(zip(lens, pos0)):
        a0, slot = int(md["cu_host"][s]), int(md["slot"][s])
        S = want[slot] * bool(p0)
        for t in range(a0, a0 + n):
            S = a6[t] * S + b6[t]
            out[t] = S
        want[slot] = S
    got = H.rglru_scan(u, g, lam, y, st, md, 8.0, torch.float32)
    close(got, out * torch.nn.functional.gelu(y6, approximate="tanh"), 2e-6)
    close(st, want, 2e-6)


# the one pass over the rows is no further from 64 bits than the row-by-row kernel (both repeat themselves exactly): rounds of 128 rows
# that end in mid-part, gates that keep little of a row's state and nearly all of it
@pytest.mark.parametrize("bias", [0.0, -2.0, -4.0])
def test_rglru_rows_are_as_exact_as_row_by_row(ops, monkeypatch, bias):
    H, _ = ops
    torch.manual_seed(5)
    lens, W = (100, 300, 413, 500, 601), 2048
    md, _, nslots = meta_of(lens, [0] * len(lens), DEV)
    T = sum(lens)
    u, g, lam, y = torch.randn(T, W, device=DEV), torch.randn(T, 2 * W, device=DEV) + bias, torch.randn(W, device=DEV), torch.randn(T, W, device=DEV)
    g6 = g.double()
    la = -8.0 * torch.sigmoid(g6[:, :W]) * torch.nn.functional.softplus(lam.double())
    a6, b6 = torch.exp(la), torch.sqrt(-torch.expm1(2 * la)) * torch.sigmoid(g6[:, W:]) * u.double()
    out, states, r = torch.empty(T, W, device=DEV).double(), [], 0
    for n in lens:
        S = torch.zeros(W, device=DEV).double()
        for t in range(r, r + n):
            S = a6[t] * S + b6[t]
            out[t] = S
        states.append(S)
        r += n
    want, err = (out * torch.nn.functional.gelu(y.double(), approximate="tanh"), torch.stack(states)), []
    monkeypatch.setattr(H, "RGLRU_ROWS", 10 ** 9)
    for m in (dict(md, q_tiles=None), md):
        st = torch.zeros(nslots, W, device=DEV)
        got = H.rglru_scan(u, g, lam, y, st, m, 8.0, torch.float32)
        err.append([float((a.double() - b).norm() / b.norm()) for a, b in zip((got, st[md["slot"].long()]), want)])
    assert err[1][0] <= 1.005 * err[0][0] and err[1][1] <= 1.01 * err[0][1], err


# more requests in a step than 16 bits count: the same rows from the one pass as row by row
def test_rglru_many_requests(ops):
    H, _ = ops
    torch.manual_seed(9)
    lens, W = [1] * 65540 + [40], 8
    md, _, nslots = meta_of(lens, [0] * len(lens), DEV)
    T = sum(lens)
    u, g, lam, y = torch.randn(T, W, device=DEV), torch.randn(T, 2 * W, device=DEV), torch.randn(W, device=DEV), torch.randn(T, W, device=DEV)
    st, st2 = torch.zeros(nslots, W, device=DEV), torch.zeros(nslots, W, device=DEV)
    got = H.rglru_scan(u, g, lam, y, st, md, 8.0, torch.float32)
    want = H.rglru_scan(u, g, lam, y, st2, dict(md, q_tiles=None), 8.0, torch.float32)
    close(got, want, 2e-6)
    close(st, st2, 2e-6)


# the chunked delta rules: chunk ends, one row and none beside long requests, a carried state, shared keys, value columns that do not fill
# four waves, decays from none to exact zeros, and (small memory) several launches that pass the state on; the oracle in fp64.  The
# bound is that of fp32 sums over some 128 terms and 16-row chains; the row-by-row kernels have to meet it too
@pytest.mark.parametrize("lens,pos0", [([24, 1, 15], [0, 3, 5]), ([16, 17, 33], [7, 0, 0]), ([150, 31], [0, 64])])
@pytest.mark.parametrize("d,dv,heads,kv,small", [(64, 64, 3, 3, False), (128, 128, 2, 1, True), (128, 48, 4, 2, False), (64, 160, 2, 2, True)])
def test_delta_chunks(ops, monkeypatch, lens, pos0, d, dv, heads, kv, small):
    H, _ = ops
    torch.manual_seed(sum(lens) + d)
    md, _, nslots = meta_of(lens, pos0, DEV)
    T, hd = sum(lens), heads * d
    f64 = lambda t, *shape: t.cpu().double().reshape(T, *shape)
    qkv, beta, gate = torch.randn(T, 2 * kv * d + heads * dv, device=DEV), torch.randn(T, heads, device=DEV), torch.randn(T, heads * dv, device=DEV)
    dec, nw = torch.rand(T, hd, device=DEV) ** 3, torch.randn(dv, device=DEV)
    dec[:, ::5], dec[:, 1::7] = 1.0, 0.0
    st = torch.randn(nslots, heads, dv, d, device=DEV)
    z, w0, nw2 = torch.randn(T, 6 * hd, device=DEV), torch.randn(hd, device=DEV) - 2.0, torch.randn(hd, device=DEV)
    r, k, v, a, wz, g = (z[:, i * hd:(i + 1) * hd] for i in range(6))
    st2 = torch.randn(nslots, heads, d, d, device=DEV)
    # fp64: gated, then generalized
    unit = lambda x, eps: x / (x.pow(2).sum(-1, keepdim=True) + eps).sqrt()
    q6 = (unit(f64(qkv[:, :kv * d], kv, d), 1e-6) * d ** -0.5).repeat_interleave(heads // kv, 1)
    k6 = unit(f64(qkv[:, kv * d:2 * kv * d], kv, d), 1e-6).repeat_interleave(heads // kv, 1)
    v6, b6, g6 = f64(qkv[:, 2 * kv * d:], heads, dv), torch.sigmoid(f64(beta, heads)), f64(dec, heads, d)
    r7, k7, v7, a7 = f64(r, heads, d), f64(k, heads, d), f64(v, heads, d), torch.sigmoid(f64(a, heads, d))
    w7, u7 = torch.exp(-0.6065 * torch.sigmoid(f64(wz, heads, d) + w0.cpu().double().reshape(heads, d))), unit(f64(k, heads, d), 1e-6)
    want, want2, o6, o7 = st.cpu().double(), st2.cpu().double(), torch.empty(T, heads, dv).double(), torch.empty(T, heads, d).double()
    for s, (n, p0) in enumerate(zip(lens, pos0)):
        a0, slot = int(md["cu_host"][s]), int(md["slot"][s])
        S, S2 = want[slot] * bool(p0), want2[slot] * bool(p0)
        for t in range(a0, a0 + n):
            S = S * g6[t][:, None, :]
            S = S + (b6[t][:, None] * (v6[t] - (S * k6[t][:, None, :]).sum(-1)))[:, :, None] * k6[t][:, None, :]
            o6[t] = (S * q6[t][:, None, :]).sum(-1)
            x = (S2 * u7[t][:, :, None]).sum(1)
            S2 = w7[t][:, :, None] * S2 - (a7[t] * u7[t])[:, :, None] * x[:, None, :] + k7[t][:, :, None] * v7[t][:, None, :]
            o7[t] = (S2 * r7[t][:, :, None]).sum(1)
        want[slot], want2[slot] = S, S2
    o6 = o6 / (o6.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * nw.cpu().double()
    o6 = o6.reshape(T, -1) * torch.sigmoid(gate.cpu().double())
    o7 = (o7 / (o7.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(T, -1) * nw2.cpu().double() * torch.sigmoid(g.cpu().double()) * 1.3
    for rows in (1, 10 ** 9):
        monkeypatch.setattr(H, "DELTA_CHUNK_ROWS", rows)
        monkeypatch.setattr(H, "GATED_CHUNK_ROWS", rows)
        if small:
            monkeypatch.setattr(H, "DELTA_FACTOR_BYTES", 4 * 4 * len(lens) * heads * (65 * d + 768))
        s1, s2 = st.clone(), st2.clone()
        got = H.gated_delta_scan(qkv, beta, dec, gate, nw, s1, md, heads, kv, d, dv, 1e-6, 1e-5, torch.float32)
        out = torch.empty(T, hd, device=DEV)
        H.delta_rule_scan(r, k, v, a, wz, g, w0, nw2, s2, md, heads, d, decay_scale=0.6065, key_eps=1e-6, norm_eps=1e-5, out_scale=1.3, out=out)
        for x, y in ((got, o6), (s1, want), (out, o7), (s2, want2)):
            close(x, y, 1e-5)


# the chunked delta rules are no further from 64 bits than the row-by-row kernels (both repeat themselves exactly; 3% for another card's sums)
@pytest.mark.parametrize("n,d", [(700, 128), (900, 64)])
@pytest.mark.parametrize("power", [3.0, 0.05])
def test_delta_chunks_are_as_exact_as_rows(ops, monkeypatch, n, d, power):
    H, _ = ops
    torch.manual_seed(n)
    h = 2
    hd, unit, f64 = h * d, lambda x: x / (x.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt(), lambda t: t.double().reshape(n, h, -1)
    md, _, nslots = meta_of([n], [0], DEV)
    qkv, beta, gate = torch.randn(n, 3 * hd, device=DEV), torch.randn(n, h, device=DEV), torch.zeros(n, hd, device=DEV)
    dec, nw = torch.rand(n, hd, device=DEV) ** power, torch.ones(d, device=DEV)
    z, w0, nw2 = torch.randn(n, 6 * hd, device=DEV), torch.randn(hd, device=DEV) - 2, torch.ones(hd, device=DEV)
    parts = [z[:, i * hd:(i + 1) * hd] for i in range(6)]
    q6, k6, v6, b6, g6 = unit(f64(qkv[:, :hd])) * d ** -0.5, unit(f64(qkv[:, hd:2 * hd])), f64(qkv[:, 2 * hd:]), torch.sigmoid(beta.double()), f64(dec)
    r7, k7, v7, a7 = f64(parts[0]), f64(parts[1]), f64(parts[2]), torch.sigmoid(f64(parts[3]))
    w7, u7 = torch.exp(-0.6065 * torch.sigmoid(f64(parts[4]) + w0.double().reshape(h, d))), unit(k7)
    S, S2 = torch.zeros(h, d, d, device=DEV).double(), torch.zeros(h, d, d, device=DEV).double()
    o6, o7 = torch.empty(n, h, d, device=DEV).double(), torch.empty(n, h, d, device=DEV).double()
    for t in range(n):
        S = S * g6[t][:, None, :]
        S = S + (b6[t][:, None] * (v6[t] - (S * k6[t][:, None, :]).sum(-1)))[:, :, None] * k6[t][:, None, :]
        o6[t] = (S * q6[t][:, None, :]).sum(-1)
        x = (S2 * u7[t][:, :, None]).sum(1)
        S2 = w7[t][:, :, None] * S2 - (a7[t] * u7[t])[:, :, None] * x[:, None, :] + k7[t][:, :, None] * v7[t][:, None, :]
        o7[t] = (S2 * r7[t][:, :, None]).sum(1)
    norm = lambda o: (o / (o.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(n, -1)
    want = (norm(o6) * 0.5, S, norm(o7) * torch.sigmoid(parts[5].double()), S2)
    err = []
    for rows in (10 ** 9, 1):
        monkeypatch.setattr(H, "DELTA_CHUNK_ROWS", rows)
        monkeypatch.setattr(H, "GATED_CHUNK_ROWS", rows)
        s1, s2, out = torch.zeros(nslots, h, d, d, device=DEV), torch.zeros(nslots, h, d, d, device=DEV), torch.empty(n, hd, device=DEV)
        got = H.gated_delta_scan(qkv, beta, dec, gate, nw, s1, md, h, h, d, d, 1e-6, 1e-5, torch.float32)
        H.delta_rule_scan(*parts, w0, nw2, s2, md, h, d, decay_scale=0.6065, key_eps=1e-6, norm_eps=1e-5, out_scale=1.0, out=out)
        slot = int(md["slot"][0])
        err.append([float((x.double() - y).norm() / y.norm()) for x, y in zip((got, s1[slot], out, s2[slot]), want)])
    assert all(c <= 1.03 * r for r, c in zip(*err)), err


# the same of the chunked delta rules: a value that is not finite changes no row before its own, no other request and no other head
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("d,heads", [(64, 2), (128, 3)])
def test_delta_chunks_values_that_are_not_finite(ops, monkeypatch, bad, d, heads):
    H, _ = ops
    torch.manual_seed(d)
    monkeypatch.setattr(H, "DELTA_CHUNK_ROWS", 1)
    monkeypatch.setattr(H, "GATED_CHUNK_ROWS", 1)
    lens, pos0 = [40, 21], [0, 5]
    md, _, nslots = meta_of(lens, pos0, DEV)
    T, hd, a1, other = sum(lens), heads * d, int(md["cu_host"][1]), int(md["slot"][1])
    qkv, beta, gate = torch.randn(T, 3 * hd, device=DEV), torch.randn(T, heads, device=DEV), torch.randn(T, hd, device=DEV)
    dec, nw = torch.rand(T, hd, device=DEV), torch.randn(d, device=DEV)
    z, w0, nw2 = torch.randn(T, 6 * hd, device=DEV), torch.randn(hd, device=DEV) - 2.0, torch.randn(hd, device=DEV)
    s0 = torch.randn(nslots, heads, d, d, device=DEV)

    def gated(qkv, beta, dec):
        st = s0.clone()
        return H.gated_delta_scan(qkv, beta, dec, gate, nw, st, md, heads, heads, d, d, 1e-6, 1e-5, torch.float32), st

    def general(z):
        st, out = s0.clone(), torch.empty(T, hd, device=DEV)
        H.delta_rule_scan(*(z[:, i * hd:(i + 1) * hd] for i in range(6)), w0, nw2, st, md, heads, d, decay_scale=0.6065, key_eps=1e-6,
                          norm_eps=1e-5, out_scale=1.3, out=out)
        return out, st

    def check(got, clean, t, row):
        assert torch.equal(got[0][:t], clean[0][:t]) and torch.equal(got[0][a1:], clean[0][a1:])
        assert torch.equal(got[0][:, d:], clean[0][:, d:])
        assert torch.equal(got[1][other], clean[1][other])
        assert not row or not bool(got[0][t, :d].isfinite().all())

    cg, cz = gated(qkv, beta, dec), general(z)
    for t in (4, 15, 20, 38):
        for at in (1, hd + 1, 2 * hd + 1):                              # of q, k and v in head 0
            x = qkv.clone()
            x[t, at] = bad
            check(gated(x, beta, dec), cg, t, True)
        x, y = beta.clone(), dec.clone()
        x[t, 0] = float("nan")
        y[t, 1] = bad
        check(gated(qkv, x, dec), cg, t, True)
        check(gated(qkv, beta, y), cg, t, t > 15)                       # (before the first rows the state is zero: inf x 0 and NaN x 0 apart)
        for i in range(6):                                              # of r, k, v, removal rate, decay and gate
            x = z.clone()
            x[t, i * hd + 1] = bad
            check(general(x), cz, t, i in (0, 1, 2) or (bad != bad and i < 5))


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("T,E,top", [(33, 10, 3), (700, 8, 2), (5, 40, 9), (300, 3, 1), (4, 8, 2), (10, 6, 3), (1, 5, 5)])
def test_routing_and_expert_products(ops, cdt, tol, T, E, top):
    H, R = ops
    torch.manual_seed(T)
    D, ff = 48, 20
    lg, corr = torch.randn(T, E, device=DEV), torch.randn(E, device=DEV) * 0.1
    a, b = H.moe_route_corrected(lg, corr, top), R.moe_route_corrected(lg, corr, top)
    assert bool((a.ids.cpu() == b.ids.cpu()).all()) and bool((a.offs.cpu() == b.offs.cpu()).all())
    # every sorted row sits in its expert's range and maps back to its token
    offs, rows, dest = a.offs.cpu().numpy(), a.rows.cpu().numpy(), a.dest.cpu().numpy()
    ids = a.ids.cpu().numpy()
    assert sorted(dest.reshape(-1).tolist()) == list(range(T * top))
    for t in range(T):
        for k in range(top):
            assert offs[ids[t, k]] <= dest[t, k] < offs[ids[t, k] + 1] and rows[dest[t, k]] == t
    close(a.w, b.w, 1e-5)
    h = torch.randn(T, D, device=DEV).to(cdt)
    wgu = torch.randn(E, 2 * ff, D, device=DEV).to(cdt)
    o1 = H.moe_weighted_sum(H.grouped_matmul_nt(H.gather_rows(h, a.rows), wgu, a.offs), a)
    o2 = R.moe_weighted_sum(R.grouped_matmul_nt(R.gather_rows(h, b.rows), wgu, b.offs), b)
    close(o1, o2, 1e-5)


# ------------------------------------------------ kernels of the latent / gated-attention / delta-rule mixers
@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_norm_offset_gate_unary_and_head_products(ops, cdt, tol):
    H, R = ops
    torch.manual_seed(3)
    x = torch.randn(37, 90, device=DEV)
    w = torch.randn(90, device=DEV) * 0.3
    close(H.group_rmsnorm(x, w, 1, 1e-5, cdt, w_offset=1.0), R.group_rmsnorm(x, w, 1, 1e-5, cdt, w_offset=1.0), tol)
    y1, y2 = torch.randn(37, 90, device=DEV), None
    a, b = x.clone(), x.clone()
    close(H.add_group_rmsnorm_(a, y1, w, 3, 1e-5, w_offset=1.0), R.add_group_rmsnorm_(b, y1, w, 3, 1e-5, w_offset=1.0), 2e-6)
    gu = torch.randn(37, 2 * 70, device=DEV) * 2
    for act in ("silu", "gelu_tanh"):
        close(H.gate_mul(gu, cdt, act), R.gate_mul(gu, cdt, act), tol)
    close(H.unary(gu[:, 3:50], "tanh", cdt), R.unary(gu[:, 3:50], "tanh", cdt), tol)
    # per-head products: heads read strided column blocks of a and write strided column blocks of out
    for T in (1, 5, 200):
        heads, K, N, a_hs, o_hs = 5, 24, 13, 30, 20
        av = torch.randn(T, heads * a_hs, device=DEV)
        wv = torch.randn(heads, N, K, device=DEV).to(cdt)
        o1 = torch.full((T, heads * o_hs), 7.0, device=DEV)
        o2 = o1.clone()
        H.head_matmul_nt(av, wv, heads, a_hs, o1, o_hs)
        R.head_matmul_nt(av, wv, heads, a_hs, o2, o_hs)
        close(o1, o2, tol)
        assert (o1[:, N:o_hs] == 7.0).all()               # columns between the heads' blocks stay untouched


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_head_norm_rope(ops, cdt, tol):
    H, R = ops
    torch.manual_seed(4)
    lens, pos0 = [1, 40, 3, 130], [900, 0, 17, 5000]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    T = sum(lens)
    for heads, n, x_col, x_hs, rot, with_w in ((3, 24, 5, 30, 10, True), (1, 14, 0, 0, 0, True), (1, 6, 14, 0, 6, False),
                                               (2, 200, 8, 200, 64, True), (4, 64, 0, 64, 64, True)):
        x = torch.randn(T, x_col + heads * max(x_hs, n) + 3, device=DEV)
        w = torch.randn(n, device=DEV) if with_w else None
        o_hs, o_col = n + 4, 2
        for paged in (False, True):
            rows = n_pages * 16 if paged else T
            outs = []
            for O in (H, R):
                out = torch.zeros(rows, o_col + heads * o_hs, device=DEV, dtype=cdt)
                raw = torch.zeros_like(out)
                O.head_norm_rope(x, heads, n, x_col, x_hs, out, o_col, o_hs, md, w=w, eps=1e-5,
                                 rot=(rot, 5000.0) if rot else None, row_map=md["kv_slot"] if paged else None, raw=raw)
                outs.append((out, raw))
            close(outs[0][0], outs[1][0], max(tol, 3e-4))     # (angles of thousands of radians in fp32)
            close(outs[0][1], outs[1][1], tol)


# heads of whole vectors (rows with all their heads in a block, angles from a table): one lane a head and all of a wave's, several rows a
# block with the last block's partly there, two vectors a lane, parts not turned, both kinds of pairs, in place, into pages, from columns
# that vectors fit (4) and do not (5: the kernel for any head).  fp32 against fp32: sums of up to 512 squares and angles of up to 6,000
# radians as products of fp32 (2^-12 of a radian at worst): 3e-4, as above; bf16 results 2^-8
@pytest.mark.parametrize("n,rot", [(4, 4), (8, 8), (20, 8), (64, 64), (64, 0), (128, 64), (132, 40), (256, 256), (260, 256), (512, 512), (512, 264)])
@pytest.mark.parametrize("heads", [1, 3, 16])
@pytest.mark.parametrize("half", [False, True])
def test_head_norm_rope_vectors(ops, n, rot, heads, half):
    H, R = ops
    torch.manual_seed(n + rot + heads)
    lens, pos0 = [1, 40, 3, 33], [900, 0, 17, 5000]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    T = sum(lens)
    for ti, to in ((torch.float32, torch.float32), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16)):
        tol = 3e-4 if to == torch.float32 else 2 ** -8
        for col, w, unit, paged, raw in ((4, True, False, False, True), (4, False, True, True, False), (5, True, True, False, False)):
            x = torch.randn(T, col + heads * (n + 8) + 3 + (5 - col) + (4 - heads * n % 4) % 4, device=DEV).to(ti)
            x = x if x.shape[1] % 4 == 0 else torch.cat([x, x[:, :4 - x.shape[1] % 4]], 1)
            wt = torch.rand(n, device=DEV) + 0.5 if w else None
            got = []
            for O in (H, R):
                out = torch.full((n_pages * 16 if paged else T, 8 + heads * (n + 4)), 3.0, device=DEV, dtype=to)
                rw = torch.zeros_like(out) if raw else None
                O.head_norm_rope(x, heads, n, col, n + 8, out, 4, n + 4, md, w=wt, eps=1e-5, rot=(rot, 5000.0) if rot else None,
                                 row_map=md["kv_slot"] if paged else None, unit_after=unit, half=half, raw=rw)
                got.append((out, rw))
            close(got[0][0], got[1][0], tol)
            assert bool((got[0][0][:, :4] == 3).all()) and bool((got[0][0][:, 4 + heads * (n + 4):] == 3).all())
            if raw:
                assert torch.equal(got[0][1], got[1][1])
            if ti == to:                                              # in place
                a, b = x.clone(), x.clone()
                for O, y in ((H, a), (R, b)):
                    O.head_norm_rope(y, heads, n, col, n + 8, y, col, n + 8, md, w=wt, eps=1e-5, rot=(rot, 5000.0) if rot else None, half=half)
                close(a, b, tol)


# a row's heads over several blocks (fewer than 1,024 rows of more heads than a block has side by side), the last block's heads fewer, a block
# that walks its heads, and rows enough for a block each; tolerance as above
@pytest.mark.parametrize("T,heads,n", [(1, 32, 512), (3, 33, 64), (300, 20, 128), (700, 48, 132), (1023, 9, 256), (1024, 9, 256)])
@pytest.mark.parametrize("half", [False, True])
def test_head_norm_rope_heads_over_blocks(ops, T, heads, n, half):
    H, R = ops
    torch.manual_seed(T + heads)
    md, _, _ = meta_of([T], [7], DEV)
    x, w = torch.randn(T, heads * n, device=DEV), torch.rand(n, device=DEV) + 0.5
    got = []
    for O in (H, R):
        out = torch.full((T, heads * n + 4), 3.0, device=DEV)
        O.head_norm_rope(x, heads, n, 0, n, out, 0, n, md, w=w, eps=1e-5, rot=(n // 16 * 8, 5000.0), half=half)
        got.append(out)
    close(got[0], got[1], 3e-4)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv,ldk,ldv,shared", [(6, 2, 24, 24, 48, 48, False), (3, 1, 20, 14, 20, 20, True),
                                                      (5, 1, 72, 56, 72, 72, True), (4, 4, 64, 64, 256, 256, False)])
def test_attention_windows_kept_tokens_and_gates(ops, cdt, tol, Hh, G, d, dv, ldk, ldv, shared):
    H, R = ops
    torch.manual_seed(5)
    lens, pos0 = [1, 70, 2, 33, 1], [150, 0, 64, 31, 3]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    T = sum(lens)
    kc = (torch.randn(n_pages, 16, ldk, device=DEV) * 0.5).to(cdt)
    vc = kc if shared else (torch.randn(n_pages, 16, ldv, device=DEV)).to(cdt)
    gb = torch.randn(Hh, device=DEV)
    for q_dt in (torch.float32, cdt):
        q = torch.randn(T, Hh * d, device=DEV).to(q_dt)
        for window, keep, gate, scale_out in ((9, 0, None, 1.0), (9, 4, None, 0.6), (40, 20, gb, 1.0), (1, 0, gb, 1.7), (40, 3, gb, 0.5),
                                              (1000, 0, None, 1.0)):
            kw = dict(scale=0.2, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=window,
                      keep_first=keep, gate_bias=gate, out_scale=scale_out)
            a = H.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw)
            b = R.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw)
            close(a, b, tol)
    # into a column block of a wider matrix
    q = torch.randn(T, Hh * d, device=DEV)
    wide = torch.zeros(T, Hh * dv + 10, device=DEV, dtype=cdt)
    kw = dict(scale=0.2, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=9, keep_first=2, gate_bias=gb)
    H.attn_paged(q, kc, vc, md, Hh, G, d, dv, out=wide[:, :Hh * dv], **kw)
    close(wide[:, :Hh * dv], R.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), tol)
    assert (wide[:, Hh * dv:] == 0).all()


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("heads,dim", [(3, 7), (2, 32), (1, 33), (4, 64), (2, 100), (3, 128), (5, 1)])
def test_input_conv_and_delta_rule_carry_state(ops, cdt, tol, heads, dim):
    H, R = ops
    torch.manual_seed(6 + dim)
    hd = heads * dim
    state = None
    for step, (lens, pos0) in enumerate((([40, 1, 3, 150], [0, 0, 0, 0]), ([1, 1, 1, 1], [40, 1, 3, 150]), ([2, 17, 1, 30], [41, 2, 4, 151]))):
        md, _, n_slots = meta_of(lens, pos0, DEV, seed=1)          # (the same slots in every step)
        T = sum(lens)
        # the input convolution: residual form, no bias, output of the GEMM type
        C = 50
        x = torch.randn(T, C, device=DEV)
        if step == 0:
            cs1 = {taps: torch.randn(n_slots, taps - 1, C, device=DEV) for taps in (1, 2, 4, 9)}
            cs2 = {taps: t.clone() for taps, t in cs1.items()}
            s1 = torch.randn(n_slots, heads, dim, dim, device=DEV)
            s2 = s1.clone()
        for taps in (1, 2, 4, 9):                                  # (nine taps: the kernel without the register window)
            cw = torch.randn(C, taps, device=DEV) * 0.5
            close(H.causal_conv(x, cw, None, cs1[taps], md, residual=True, out_dtype=cdt),
                  R.causal_conv(x, cw, None, cs2[taps], md, residual=True, out_dtype=cdt), tol)
            if taps > 1:
                close(cs1[taps][md["slot"].long()], cs2[taps][md["slot"].long()], 1e-6)
        z = torch.randn(T, 6 * hd + 5, device=DEV)
        r, k, v, a, wz, g = (z[:, i * hd:(i + 1) * hd] for i in range(6))
        w0, nw = torch.randn(hd, device=DEV) - 2.0, torch.randn(hd, device=DEV)
        o1 = torch.zeros(T, hd + 3, device=DEV, dtype=cdt)
        o2 = torch.zeros_like(o1)
        kw = dict(decay_scale=0.6065, key_eps=1e-6, norm_eps=1e-5, out_scale=1.3)
        H.delta_rule_scan(r, k, v, a, wz, g, w0, nw, s1, md, heads, dim, out=o1[:, :hd], **kw)
        R.delta_rule_scan(r, k, v, a, wz, g, w0, nw, s2, md, heads, dim, out=o2[:, :hd], **kw)
        close(o1, o2, max(tol, 2e-4))
        close(s1[md["slot"].long()], s2[md["slot"].long()], 2e-4)


@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (128, 64)])
def test_matrix_core_attention_over_row_tiles(ops, d, dv):
    """bf16 prompts of several 128-row tiles through the matrix-core kernel (fp32 and bf16 queries):
    windows shorter and longer than a tile, kept first keys filling more than one key tile, sigmoid
    gates, pool rows wider than the heads, and a step-local table of one-row pages."""
    H, R = ops
    torch.manual_seed(8)
    cdt = torch.bfloat16
    Hh, G = 4, 2
    lens, pos0 = [300, 17, 129], [0, 0, 0]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    T = sum(lens)
    kc = (torch.randn(n_pages, 16, G * d + 16, device=DEV) * 0.5).to(cdt)
    vc = torch.randn(n_pages, 16, G * dv + 8, device=DEV).to(cdt)
    gb = torch.randn(Hh, device=DEV)
    for q_dt in (torch.float32, cdt):
        q = torch.randn(T, Hh * d, device=DEV).to(q_dt)
        for window, keep, gate in ((40, 0, None), (40, 50, None), (200, 70, gb), (7, 3, gb), (1000, 0, gb)):
            kw = dict(scale=d ** -0.5, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=window,
                      keep_first=keep, gate_bias=gate, out_scale=0.8)
            close(H.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), R.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), 2e-2)
    # keys and values of the step itself, one row a page, every head its own
    cu = md["cu_host"]
    local = torch.from_numpy((cu[:-1, None] + np.arange(max(lens))[None, :]).astype(np.int32)).to(DEV)
    kf = (torch.randn(T, 1, Hh * d, device=DEV) * 0.5).to(cdt)
    vf = torch.randn(T, 1, Hh * dv, device=DEV).to(cdt)
    q = torch.randn(T, Hh * d, device=DEV)
    kw = dict(scale=d ** -0.5, softcap=0.0, r1=None, r2=None, chunk=0, page_size=1, out_dtype=cdt, window=33)
    lm = dict(md, page_table=local)
    close(H.attn_paged(q, kf, vf, lm, Hh, Hh, d, dv, **kw), R.attn_paged(q, kf, vf, lm, Hh, Hh, d, dv, **kw), 2e-2)


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_decode_rows_over_long_contexts_split_their_keys(ops, cdt, tol):
    """Three decode rows far into their sequences: the launch cuts every row's keys into ranges that run
    as blocks of their own and merges them (softmax parts by their maxima and sums, gated parts by
    addition); a row near the start has ranges without keys."""
    H, R = ops
    torch.manual_seed(9)
    lens, pos0 = [1, 1, 1], [1500, 3, 700]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    Hh, G, d, dv = 4, 2, 24, 40
    kc = (torch.randn(n_pages, 16, G * d, device=DEV) * 0.5).to(cdt)
    vc = torch.randn(n_pages, 16, G * dv, device=DEV).to(cdt)
    q = torch.randn(3, Hh * d, device=DEV)
    gb = torch.randn(Hh, device=DEV)
    for window, keep, gate in ((0, 0, None), (1000, 0, None), (600, 90, gb), (0, 0, gb)):
        kw = dict(scale=0.3, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=window,
                  keep_first=keep, gate_bias=gate, out_scale=0.9)
        close(H.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), R.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), tol)


@pytest.mark.parametrize("d,dv,Hh", [(192, 128, 5), (320, 256, 32), (576, 512, 16)])
def test_heads_of_a_token_share_one_matrix_core_tile(ops, d, dv, Hh):
    """Decode rows over latent rows (one key / value head, values = the first columns of the key rows):
    the kernel that takes a token's heads as the columns of one tile, with the keys cut over several
    blocks and merged, rows with fewer keys than a tile, windows and kept first keys."""
    H, R = ops
    torch.manual_seed(10)
    cdt = torch.bfloat16
    lens, pos0 = [1, 1, 1, 1], [1500, 3, 700, 31]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    pool = (torch.randn(n_pages, 16, d, device=DEV) * 0.3).to(cdt)
    q = torch.randn(4, Hh * d, device=DEV)
    for window, keep in ((0, 0), (1000, 0), (600, 90), (33, 0)):
        kw = dict(scale=d ** -0.5, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=window,
                  keep_first=keep, out_scale=0.9)
        close(H.attn_paged(q, pool, pool, md, Hh, 1, d, dv, **kw), R.attn_paged(q, pool, pool, md, Hh, 1, d, dv, **kw), 2e-2)


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_dyt_norm_scaled_add_and_embedding_scale(ops, cdt, tol):
    """Dynamic Tanh norm (vector path and odd widths, row gather, column slices), x += m y, embedding rows times a scale."""
    H, R = ops
    torch.manual_seed(11)
    for T, D in ((7, 320), (3, 37), (130, 2048), (1, 4100)):
        x = torch.randn(T, D + 8, device=DEV)[:, 4:4 + D] * 2
        wb = torch.randn(2, D, device=DEV)
        alpha = torch.tensor([0.7], device=DEV)
        close(H.dyt_norm(x, wb, alpha, cdt), R.dyt_norm(x, wb, alpha, cdt), tol)
        xc = x.contiguous()
        close(H.dyt_norm(xc, wb, alpha, cdt), R.dyt_norm(xc, wb, alpha, cdt), tol)
        idx = torch.tensor([T - 1, 0, T // 2], dtype=torch.int32, device=DEV)
        close(H.dyt_norm(xc, wb, alpha, torch.float32, row_idx=idx), R.dyt_norm(xc, wb, alpha, torch.float32, row_idx=idx), 1e-5)
        y = torch.randn(T, D, device=DEV)
        a, b = xc.clone(), xc.clone()
        close(H.add_scaled_(a, y, 0.6), R.add_scaled_(b, y, 0.6), 1e-6)
        ys = torch.randn(T, D + 3, device=DEV)[:, 1:1 + D]
        close(H.add_scaled_(a, ys, -1.3), R.add_scaled_(b, ys, -1.3), 1e-6)
    table = torch.randn(50, 36, device=DEV).to(cdt)
    ids = torch.tensor([3, 49, 0, 3], dtype=torch.int32, device=DEV)
    close(H.embed_rows(ids, table, scale=0.37), R.embed_rows(ids, table, scale=0.37), 1e-6)


# entries to their experts' rows, counted by the placement itself (up to 2,048 entries of 16 experts) and from counts: one block and several, wave and block edges, one expert and
# the most, one that nobody takes; every entry in its expert's range, once
@pytest.mark.parametrize("T,top", [(65, 1), (127, 2), (512, 2), (513, 2), (512, 4), (513, 4), (1500, 1), (2048, 1), (2049, 1)])
@pytest.mark.parametrize("E", [1, 8, 10, 16, 17, 130])
def test_placement_counts_itself(ops, T, top, E):
    H, R = ops
    if top > E:
        return
    torch.manual_seed(T + E)
    logits = torch.randn(T, E, device=DEV)
    logits[:, E // 2:E // 2 + 1] -= 50.0 if E > top else 0.0                     # (an expert that nobody takes)
    for r in (H.moe_route_softmax_grouped(logits, None, top, 0, 0, 1.0), H.moe_route_corrected(logits, torch.zeros(E, device=DEV), top),
              H.moe_route_corrected(logits, None, top), H.moe_route_grouped(logits, top, 0, 0, 1.0)):
        ids = r.ids.long().flatten().cpu()
        assert torch.equal(r.offs.long().cpu(), torch.cat([torch.zeros(1, dtype=torch.long), torch.bincount(ids, minlength=E).cumsum(0)]))
        dest = r.dest.long().flatten().cpu()
        assert torch.equal(dest.sort().values, torch.arange(T * top))
        assert torch.equal(torch.bucketize(dest, r.offs.long().cpu()[1:], right=True), ids)
        assert torch.equal(r.rows.long().cpu()[dest], torch.arange(T).repeat_interleave(top))


# no tokens: no rows of any expert, whatever the memory held
@pytest.mark.parametrize("E", [8, 40])
def test_routes_of_no_tokens(ops, E):
    H, _ = ops
    logits = torch.randn(0, E, device=DEV)
    for route in (lambda: H.moe_route_softmax_grouped(logits, None, 2, 0, 0, 1.0), lambda: H.moe_route_grouped(logits, 2, 0, 0, 1.0),
                  lambda: H.moe_route_corrected(logits, torch.zeros(E, device=DEV), 2), lambda: H.moe_route_corrected(logits, None, 2)):
        junk = torch.full((E + 1,), 7, dtype=torch.int32, device=DEV)
        del junk
        r = route()
        assert r.offs.shape == (E + 1,) and not bool(r.offs.any()) and r.dest.shape == (0, 2) and r.rows.numel() == 0


# gathered rows by 16 bytes and by elements: the same bytes, for widths about a block's threads, column slices and rows that vectors do not fit
@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D", [8, 36, 512, 520, 1032, 2056, 4])
def test_gathered_rows(ops, cdt, D):
    H, _ = ops
    x = torch.randn(50, D + 16, device=DEV).to(cdt)
    idx = torch.tensor([49, 0, 7, 7, 31], dtype=torch.int32, device=DEV)
    for a in (x[:, :D], x[:, 8:8 + D], x[:, 1:1 + D], x[:, :D].contiguous()):
        assert torch.equal(H.gather_rows(a, idx), a[idx.long()])


# embedding rows by four columns a lane and by one: widths about a block's turn of 1,024 columns and the four or two of them in flight, tables that vectors do
# not fit; ids out of range; with positions, pairs and copies.  Sums of three values of the table's type in fp32, whose order is the oracle's: 1e-6
@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D", [4, 1020, 1024, 1028, 2052, 4096, 4100, 1023])
def test_embedding_widths(ops, cdt, D):
    H, R = ops
    torch.manual_seed(D)
    flat = torch.randn(60 * D + 1, device=DEV).to(cdt)
    ids = torch.tensor([3, 59, 0, 77, -1, 12], dtype=torch.int32, device=DEV)
    clamped = ids.clamp(0, 59)
    for table in (flat[:60 * D].view(60, D), flat[1:].view(60, D)):
        close(H.embed_rows(ids, table, scale=0.37), R.embed_rows(clamped, table, scale=0.37), 1e-6)
        ptab, pairs = torch.randn(9, D, device=DEV).to(cdt), torch.randn(12, D, device=DEV).to(cdt)
        pos, prev = torch.arange(6, dtype=torch.int32, device=DEV), torch.tensor([-1, 3, 4, 0, 9, 50], dtype=torch.int32, device=DEV)
        for kw in (dict(pos_table=ptab, tok_pos=pos), dict(bigram=(pairs, prev, 31, 17)), dict(pos_table=ptab, tok_pos=pos, copies=3)):
            close(H.embed_rows(ids, table, **kw), R.embed_rows(clamped, table, **kw), 1e-6)


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_rotation_with_rescaled_frequencies_then_unit_norm(ops, cdt, tol):
    """Pair rotation with wavelength-rescaled frequencies followed by the weightless RMS norm, into rows and into pools;
    a plain placement (no norm, no rotation) of value heads."""
    H, R = ops
    torch.manual_seed(12)
    lens, pos0 = [1, 40, 3, 130], [900, 0, 17, 2000]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    T = sum(lens)
    sc = (8.0, 1.0, 4.0, 64)
    f = R.rope_freqs(16, 100.0, "cpu", sc).double()
    f0 = R.rope_freqs(16, 100.0, "cpu").double()
    ratio = (f / f0).numpy()
    assert ratio[0] == 1.0 and abs(ratio[-1] - 1 / 8) < 1e-6 and ((ratio[1:] <= ratio[:-1] + 1e-9).all())   # kept, blended, slowed
    assert ((ratio > 1 / 8 + 1e-3) & (ratio < 1 - 1e-3)).any()
    for heads, n, x_col, rot in ((3, 24, 5, (16, 100.0, sc)), (2, 40, 0, (40, 30000.0, (4.0, 2.0, 8.0, 512))), (4, 64, 0, (32, 1e4, None)),
                                 (1, 6, 2, None), (2, 130, 0, (128, 500.0, None))):
        x = torch.randn(T, x_col + heads * n + 3, device=DEV) * 3
        for paged in (False, True):
            rows = n_pages * 16 if paged else T
            outs = []
            for O in (H, R):
                out = torch.zeros(rows, heads * n, device=DEV, dtype=cdt)
                O.head_norm_rope(x, heads, n, x_col, n, out, 0, n, md, eps=1e-5, rot=rot, unit_after=True,
                                 row_map=md["kv_slot"] if paged else None)
                outs.append(out)
            close(outs[0], outs[1], max(tol, 3e-4))
            if not paged:                                       # every head has unit mean square
                ms = outs[0].float().view(T, heads, n).pow(2).mean(-1)
                assert (ms - 1).abs().max().item() < (2e-2 if cdt == torch.bfloat16 else 1e-3)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv", [(5, 5, 40, 72), (6, 2, 24, 40), (4, 2, 64, 64), (8, 2, 128, 128), (4, 4, 128, 64), (3, 1, 20, 14)])
def test_attention_with_a_silent_softmax_entry_and_head_gates(ops, cdt, tol, Hh, G, d, dv):
    """Windowed softmax with one more entry of a given score and no value, and a sigmoid gate per (row, head): prompts
    (per-row kernel, and row tiles on the matrix cores where the head sizes allow), portions, decode rows."""
    H, R = ops
    torch.manual_seed(13)
    lens, pos0 = [1, 170, 2, 33, 1], [150, 0, 64, 31, 3]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    T = sum(lens)
    kc = (torch.randn(n_pages, 16, G * d, device=DEV) * 0.5).to(cdt)
    vc = torch.randn(n_pages, 16, G * dv, device=DEV).to(cdt)
    z = torch.randn(T, Hh * d + Hh + 5, device=DEV)
    hg = z[:, Hh * d:Hh * d + Hh]                               # a column block of a wider matrix
    q = torch.randn(T, Hh * d, device=DEV) * (8 / d) ** 0.5      # (scores of a few units whatever the head size)
    for window, sink, gate, scale in ((9, 0.0, hg, 0.2), (72, 0.0, hg, 0.5), (72, 1.5, None, 0.2), (1, 0.0, hg, 0.3), (0, -2.0, hg, 0.05),
                                      (40, None, hg, 0.2), (40, 0.0, hg, 1.5), (40, 0.0, hg, -1.5)):
        kw = dict(scale=scale, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=window, sink=sink,
                  head_gate=gate)
        a = H.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw)
        b = R.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw)
        close(a, b, tol)
    # decode rows far into their sequences: every row's keys cut over blocks, the silent entry joins once in the merge
    lens, pos0 = [1, 1, 1], [1500, 3, 700]
    md, n_pages, _ = meta_of(lens, pos0, DEV)
    kc = (torch.randn(n_pages, 16, G * d, device=DEV) * 0.5).to(cdt)
    vc = torch.randn(n_pages, 16, G * dv, device=DEV).to(cdt)
    q = torch.randn(3, Hh * d, device=DEV) * (8 / d) ** 0.5
    hg = torch.randn(3, Hh, device=DEV)
    for window, sink, scale in ((0, 0.0, 0.3), (1000, 0.0, 0.01), (1000, 3.0, 0.3), (600, 0.0, -1.0)):
        kw = dict(scale=scale, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=window, sink=sink, head_gate=hg)
        close(H.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), R.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), tol)


@pytest.mark.parametrize("T,E,top", [(33, 10, 3), (700, 8, 2), (5, 40, 9), (300, 3, 1), (4, 8, 8), (1, 5, 5)])
def test_topk_routing_and_combine(ops, T, E, top):
    """The largest logits choose, the softmax over the chosen weighs; the combine adds the weighted expert rows, the gated
    shared expert's row and the residual in one pass."""
    H, R = ops
    torch.manual_seed(14)
    D = 52
    z = torch.randn(T, E + 3, device=DEV)
    logits = z[:, 1:1 + E]
    a, b = H.moe_route_topk(logits, top), R.moe_route_topk(logits, top)
    assert torch.equal(a.ids.cpu().long(), b.ids.cpu().long())
    close(a.w, b.w, 1e-5)
    assert (a.w.sum(-1) - 1).abs().max().item() < 1e-5
    assert torch.equal(a.offs.cpu().long(), b.offs.cpu().long())
    # a tie goes to the lower expert
    tie = torch.zeros(2, E, device=DEV)
    assert H.moe_route_topk(tie, top).ids.cpu().tolist() == [list(range(top))] * 2
    y = torch.randn(T * top, D, device=DEV)
    shared = torch.randn(T, D, device=DEV)
    gate = torch.randn(T, 4, device=DEV)[:, 2:3]
    for sh, g in ((None, None), (shared, gate), (shared, None)):
        x1, x2 = torch.randn(T, D, device=DEV), None
        x2 = x1.clone()
        H.moe_combine_(x1, y, a, 0.6, sh, g)
        R.moe_combine_(x2, y, a, 0.6, sh, g)
        close(x1, x2, 1e-5)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv,taps,rot", [(6, 2, 24, 40, 3, (16, 100.0, (8.0, 1.0, 4.0, 64))), (3, 3, 40, 72, 4, (40, 3e4, None)),
                                                (4, 0, 64, 64, 2, (32, 1e4, None)), (2, 1, 128, 96, 1, (128, 5e5, None)),
                                                (2, 2, 10, 6, 10, None), (5, 1, 130, 200, 5, (64, 1e3, None))])
def test_projected_rows_into_attention_in_one_pass(ops, cdt, tol, Hh, G, d, dv, taps, rot):
    """Convolution with carried history, rotation, unit norm and page write of q | k | v rows as one kernel against the
    chain of plain ops: prompts, portions that continue a request, single decoded rows (which also rewrite the history),
    query-only layers (G = 0), one tap, no convolution at all."""
    H, R = ops
    torch.manual_seed(15)
    C = Hh * d + G * (d + dv)
    for lens, pos0 in (([1, 40, 3, 130], [900, 0, 17, 2000]), ([1, 1, 1], [5, 0, 300])):
        md, n_pages, n_slots = meta_of(lens, pos0, DEV)
        T = sum(lens)
        z = torch.randn(T, C + Hh + 3, device=DEV)
        for w in ((torch.randn(C, taps, device=DEV) * 0.5), None):
            st0 = torch.randn(n_slots, taps - 1, C, device=DEV) if (w is not None and taps > 1) else None
            outs = []
            for O in (H, R):
                st = st0.clone() if st0 is not None else None
                q = torch.zeros(T, Hh * d, device=DEV)
                kc = torch.zeros(n_pages, 16, max(G, 1) * d, device=DEV, dtype=cdt)
                vc = torch.zeros(n_pages, 16, max(G, 1) * dv, device=DEV, dtype=cdt)
                O.qkv_conv_rope_store(z, w, st, md, Hh, G, d, dv, q, kc if G else None, vc if G else None, eps=1e-5, rot=rot)
                outs.append((q, kc, vc, st))
            close(outs[0][0], outs[1][0], 3e-4)
            close(outs[0][1], outs[1][1], max(tol, 3e-4))
            close(outs[0][2], outs[1][2], tol) if G else None
            if st0 is not None:
                used = md["slot"].long()
                close(outs[0][3][used], outs[1][3][used], 1e-6)
                free = [i for i in range(n_slots) if i not in used.tolist()]
                assert torch.equal(outs[0][3][free], st0[free])


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_residual_add_with_the_next_norm(ops, cdt, tol):
    H, R = ops
    torch.manual_seed(16)
    for T, D in ((7, 320), (3, 37), (130, 2048)):
        x = torch.randn(T, D, device=DEV) * 2
        y = torch.randn(T, D + 4, device=DEV)[:, 2:2 + D]
        wb, alpha = torch.randn(2, D, device=DEV), torch.tensor([0.6], device=DEV)
        a, b = x.clone(), x.clone()
        ha, hb = H.add_scaled_dyt_norm_(a, y, 0.6, wb, alpha, cdt), R.add_scaled_dyt_norm_(b, y, 0.6, wb, alpha, cdt)
        close(a, b, 1e-6)
        close(ha, hb, tol)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("S,D", [(1, 36), (3, 320), (5, 34), (2, 2304)])
def test_residual_streams_norm_update_and_embedding_copies(ops, cdt, tol, S, D):
    """Several residual streams side by side in a row: their weighted sum through the RMS norm (also the plain
    sum with a row gather), the update of all streams at once with the gated sublayer output (gate logits as a
    column block of a wider matrix), the same fused with the next norm, one stream without coefficients, and the
    embedding with a position vector written S times."""
    H, R = ops
    torch.manual_seed(S * D)
    T = 37
    xs = torch.randn(T, S * D, device=DEV)
    hc = torch.randn(2 * S + S * S, device=DEV)
    w = 1 + 0.3 * torch.randn(D, device=DEV)
    idx = torch.tensor([5, 0, 36, 5], dtype=torch.int32, device=DEV)
    close(H.streams_norm(xs, hc, w, 1e-5, cdt, S), R.streams_norm(xs, hc, w, 1e-5, cdt, S), tol)
    close(H.streams_norm(xs, None, w, 1e-5, cdt, S, row_idx=idx), R.streams_norm(xs, None, w, 1e-5, cdt, S, row_idx=idx), tol)
    y = torch.randn(T, D, device=DEV)
    z = torch.randn(T, D + 24, device=DEV)
    gate = z[:, 8:8 + D]
    for g in (gate, None):
        a, b = xs.clone(), xs.clone()
        close(H.streams_update_(a, y, g, hc, 0.45, S), R.streams_update_(b, y, g, hc, 0.45, S), 1e-5)
        a, b = xs.clone(), xs.clone()
        hc2 = torch.randn(2 * S + S * S, device=DEV)
        close(H.streams_update_norm_(a, y, g, hc, 0.45, S, hc2, w, 1e-5, cdt), R.streams_update_norm_(b, y, g, hc, 0.45, S, hc2, w, 1e-5, cdt), tol)
        close(a, b, 1e-5)
    if S == 1:
        a, b = xs.clone(), xs.clone()
        close(H.streams_update_norm_(a, y, gate, None, 0.7, 1, None, w, 1e-5, cdt), R.streams_update_norm_(b, y, gate, None, 0.7, 1, None, w, 1e-5, cdt), tol)
        close(a, b, 1e-5)
    table, ptab = torch.randn(50, D, device=DEV).to(cdt), torch.randn(90, D, device=DEV).to(cdt)
    ids = torch.randint(0, 50, (T,), dtype=torch.int32, device=DEV)
    pos = torch.randint(0, 90, (T,), dtype=torch.int32, device=DEV)
    close(H.embed_rows(ids, table, pos_table=ptab, tok_pos=pos, copies=S), R.embed_rows(ids, table, pos_table=ptab, tok_pos=pos, copies=S), 1e-6)
    close(H.embed_rows(ids, table, scale=1.5, copies=S), R.embed_rows(ids, table, scale=1.5, copies=S), 1e-6)
    lg, eye = torch.randn(T, 70, device=DEV), torch.eye(70, device=DEV)
    close(H.matmul_nt(lg, eye, scale=0.25), R.matmul_nt(lg, eye, scale=0.25), 1e-7)
    o = torch.randn(T, D, device=DEV)
    close(H.sigmoid_gate(o, y, cdt), R.sigmoid_gate(o, y, cdt), tol)
    close(H.sigmoid_gate(o.to(cdt), y, cdt), R.sigmoid_gate(o.to(cdt), y, cdt), tol)
    close(H.unary(o, "gelu", cdt), R.unary(o, "gelu", cdt), tol)


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_rotation_in_halves_with_turn_count_rescaling(ops, cdt, tol):
    """Pairs (i, i + dims / 2) with frequencies rescaled by turn counts and amplified cosines and sines, with and
    without the norm in front, over part of a head and over heads wider than a wave, into a pool and in place."""
    H, R = ops
    torch.manual_seed(4)
    md, n_pages, _ = meta_of([40, 3, 1], [0, 77, 1200], DEV)
    T = 44
    sc = ("turns", 3.0, 300.0, 20.0, 2.0)
    for heads, n, dims in ((3, 32, 32), (2, 24, 10), (1, 200, 160), (4, 8, 8)):
        x = torch.randn(T, heads * n + 6, device=DEV)
        w = 1 + 0.2 * torch.randn(n, device=DEV)
        for ww in (w, None):
            a, b = torch.zeros(T, heads * n, device=DEV, dtype=cdt), torch.zeros(T, heads * n, device=DEV, dtype=cdt)
            kw = dict(w=ww, eps=1e-5, rot=(dims, 1e4, sc), half=True)
            close(H.head_norm_rope(x, heads, n, 3, n, a, 0, n, md, **kw), R.head_norm_rope(x, heads, n, 3, n, b, 0, n, md, **kw), tol)
        pa = torch.zeros(n_pages * 16, n + 5, device=DEV, dtype=cdt)
        pb = pa.clone()
        kw = dict(rot=(dims, 1e4, sc), half=True, row_map=md["kv_slot"])
        close(H.head_norm_rope(x, 1, n, 0, 0, pa, 5, 0, md, **kw), R.head_norm_rope(x, 1, n, 0, 0, pb, 5, 0, md, **kw), tol)
        xa, xb = x.clone(), x.clone()                                   # in place: every pair is read before it is written
        kw = dict(rot=(dims, 50.0), half=True)
        close(H.head_norm_rope(xa, heads, dims, n - dims, n, xa, n - dims, n, md, **kw), R.head_norm_rope(xb, heads, dims, n - dims, n, xb, n - dims, n, md, **kw), 1e-5)
    f = R.rope_freqs(32, 1e6, "cpu", sc)
    f0 = R.rope_freqs(32, 1e6, "cpu")
    assert f[0] == f0[0] and abs(float(f[-1] / f0[-1]) - 1 / 3) < 1e-6 and abs(R.rope_amp(sc) - (0.1 * np.log(3.0) + 1)) < 1e-12


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv", [(6, 2, 10, 14), (2, 2, 32, 48), (4, 2, 64, 128), (2, 1, 128, 64)])
def test_two_score_maps_over_shared_values_and_their_combine(ops, cdt, tol, Hh, G, d, dv):
    """Differential attention's pieces: 2 H query heads over 2 G key heads whose value head is the key head
    modulo G, fp32 outputs over pools of the GEMM type (prompt rows over tiles and decoded rows over long
    contexts with split keys), then the combine a1 - lambda a2 with its unit norm."""
    H, R = ops
    torch.manual_seed(Hh * d)
    for lens, pos0 in (([150, 17], [0, 0]), ([1, 1], [700, 45]), ([5, 40], [3, 90])):
        md, n_pages, _ = meta_of(lens, pos0, DEV)
        T = sum(lens)
        kc = (torch.randn(n_pages, 16, 2 * G * d, device=DEV) * 0.5).to(cdt)
        vc = torch.randn(n_pages, 16, G * dv, device=DEV).to(cdt)
        q = torch.randn(T, 2 * Hh * d, device=DEV)
        kw = dict(scale=d ** -0.5, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, v_heads=G)
        a, b = torch.empty(T, 2 * Hh * dv, device=DEV), torch.empty(T, 2 * Hh * dv, device=DEV)
        H.attn_paged(q, kc, vc, md, 2 * Hh, 2 * G, d, dv, out=a, **kw)
        R.attn_paged(q, kc, vc, md, 2 * Hh, 2 * G, d, dv, out=b, **kw)
        close(a, b, 2e-5 if cdt == torch.float32 else 1e-2)
        lam = 0.4 * torch.randn(4, d, device=DEV)
        close(H.diff_combine(b, lam, 0.35, Hh, dv, 1e-6, cdt), R.diff_combine(b, lam, 0.35, Hh, dv, 1e-6, cdt), tol)


@pytest.mark.parametrize("heads,dim,vdim", [(3, 7, 9), (5, 48, 72), (1, 1, 1), (2, 130, 70), (4, 128, 128), (1, 256, 300)])
def test_hgrn2_scan_carries_state(ops, heads, dim, vdim):
    """The gated recurrence over a batch of unequal requests, some continuing from carried states in scattered
    slots (prompt portions and single decoded rows), with and without the gate's bias; outputs and states."""
    H, R = ops
    torch.manual_seed(heads + dim)
    for lens, pos0 in (([33, 1, 7], [0, 5, 12]), ([1, 1, 1], [4, 0, 9]), ([70], [0])):
        md, _, n_slots = meta_of(lens, pos0, DEV)
        T = sum(lens)
        z = torch.randn(T, 2 * heads * dim + heads * vdim + 5, device=DEV)
        q, f, v = z[:, :heads * dim], z[:, heads * dim:2 * heads * dim], z[:, 2 * heads * dim:2 * heads * dim + heads * vdim]
        fb = torch.randn(heads * dim, device=DEV)
        lower = torch.rand(heads * dim, device=DEV)
        nw = 1 + 0.2 * torch.randn(vdim, device=DEV)
        st = torch.randn(n_slots, heads, dim, vdim, device=DEV)
        for bias in (fb, None):
            s1, s2 = st.clone(), st.clone()
            a = H.hgrn2_scan(q, f, v, bias, lower, nw, s1, md, heads, dim, vdim, 1e-5, torch.float32)
            b = R.hgrn2_scan(q, f, v, bias, lower, nw, s2, md, heads, dim, vdim, 1e-5, torch.float32)
            close(a, b, 2e-4)
            close(s1[md["slot"].long()], s2[md["slot"].long()], 2e-4)


@pytest.mark.parametrize("T,E,top,groups,keep", [(50, 8, 2, 4, 3), (7, 12, 3, 4, 2), (300, 5, 2, 5, 3), (33, 6, 6, 2, 2), (20, 7, 1, 0, 0),
                                                 (64, 64, 8, 8, 4), (9, 128, 16, 64, 9)])
def test_grouped_sigmoid_routing(ops, T, E, top, groups, keep):
    H, R = ops
    torch.manual_seed(T + E)
    logits = torch.randn(T, E + 3, device=DEV)[:, 1:1 + E] * 2
    a, b = H.moe_route_grouped(logits, top, groups, keep, 1.9), R.moe_route_grouped(logits, top, groups, keep, 1.9)
    assert torch.equal(a.ids.cpu().sort(-1).values, b.ids.cpu().sort(-1).values)
    assert torch.equal(a.ids.cpu(), b.ids.cpu())
    close(a.w, b.w, 1e-5)
    assert torch.equal(a.offs.cpu(), b.offs.cpu())
    assert torch.equal(a.rows.cpu().long().bincount(minlength=T), torch.full((T,), top))
    # every (token, choice) sits in its expert's range of sorted rows
    offs, dest = a.offs.cpu().long(), a.dest.cpu().long()
    assert bool(((dest >= offs[a.ids.cpu().long()]) & (dest < offs[a.ids.cpu().long() + 1])).all())
    assert torch.equal(a.rows.cpu().long()[dest], torch.arange(T)[:, None].expand(T, top))


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,Gv,d,dv,rot", [(12, 4, 2, 10, 14, (6, 50.0)), (8, 4, 2, 64, 128, (32, 1e6)), (2, 2, 1, 32, 64, (32, 1e4)),
                                              (4, 2, 1, 130, 70, None)])
def test_projected_rows_with_weighted_norms_before_the_rotation(ops, cdt, tol, Hh, G, Gv, d, dv, rot):
    """The one-pass kernel in its second form: q and k heads RMS-normed with a weight before the rotation, fewer
    value heads than key heads in the row, no convolution; against the chain of plain ops."""
    H, R = ops
    torch.manual_seed(21)
    C = Hh * d + G * d + Gv * dv
    qw, kw_ = 1 + 0.3 * torch.randn(d, device=DEV), 1 + 0.3 * torch.randn(d, device=DEV)
    for lens, pos0 in (([1, 40, 3, 130], [900, 0, 17, 2000]), ([1, 1, 1], [5, 0, 300])):
        md, n_pages, _ = meta_of(lens, pos0, DEV)
        T = sum(lens)
        z = torch.randn(T, C + 7, device=DEV)
        outs = []
        for O in (H, R):
            q = torch.zeros(T, Hh * d, device=DEV)
            kc = torch.zeros(n_pages, 16, G * d, device=DEV, dtype=cdt)
            vc = torch.zeros(n_pages, 16, Gv * dv, device=DEV, dtype=cdt)
            O.qkv_conv_rope_store(z, None, None, md, Hh, G, d, dv, q, kc, vc, eps=1e-5, rot=rot, v_heads=Gv, q_norm=qw, k_norm=kw_)
            outs.append((q, kc, vc))
        close(outs[0][0], outs[1][0], 3e-4)
        close(outs[0][1], outs[1][1], max(tol, 3e-4))
        close(outs[0][2], outs[1][2], tol)


def blocks_of(lens, pos0, P, ps, dev, kcols, vcols, cdt, seed=3):
    """Block pools in scattered pages: (block keys, block values, table, P), garbage where nothing is written."""
    rng = np.random.default_rng(seed)
    need = [max(1, -(-((p + n) // P) // ps)) for p, n in zip(pos0, lens)]
    tab = np.full((len(lens), max(need)), -1, np.int32)
    perm = rng.permutation(sum(need) + 3)
    k = 0
    for b, m in enumerate(need):
        tab[b, :m] = perm[k:k + m]
        k += m
    pools = [torch.randn(sum(need) + 3, ps, c, device=dev).to(cdt) for c in (kcols, vcols)]
    return pools[0], pools[1], torch.from_numpy(tab).to(dev), P


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("P", [1, 3, 16, 40])
@pytest.mark.parametrize("kcols,vcols", [(20, 14), (64, 128), (200, 36)])
def test_block_means(ops, cdt, tol, P, kcols, vcols):
    """Blocks completed by whole prompts, by portions that begin inside a block, and by single rows; rows of the
    block pools that no completed block owns stay as they were."""
    H, R = ops
    torch.manual_seed(P + kcols)
    for lens, pos0 in (([70, 5, 33], [0, 0, 0]), ([3, 40, 1], [70, 5, 33]), ([1, 1, 1], [39, 2, 15]), ([2, 2], [38, 0])):
        md, npages, _ = meta_of(lens, pos0, DEV)
        kc, vc = torch.randn(npages, 16, kcols, device=DEV).to(cdt), torch.randn(npages, 16, vcols, device=DEV).to(cdt)
        b1 = blocks_of(lens, pos0, P, 16, DEV, kcols, vcols, cdt)
        b2 = (b1[0].clone(), b1[1].clone()) + b1[2:]
        H.block_means(kc, vc, b1, md, kcols, vcols)
        R.block_means(kc, vc, b2, md, kcols, vcols)
        for x, y in zip(b1[:2], b2[:2]):
            close(x, y, 1e-6 if cdt == torch.float32 else 8e-3)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv,rot", [(6, 2, 10, 14, (6, 50.0, ("turns", 3.0, 24.0, 4.0, 0.5))), (8, 4, 64, 128, (64, 1e6, None)),
                                           (4, 2, 128, 128, (128, 5e5, ("turns", 8.0, 128.0, 16.0, 1.0))), (2, 1, 96, 96, (96, 1e4, None)),
                                           (2, 2, 150, 130, (140, 1e4, ("turns", 2.0, 64.0, 8.0, 1.0))), (3, 1, 300, 40, (20, 1e3, None)),
                                           (3, 3, 8, 5, None)])
def test_projected_rows_rotated_in_halves_with_block_means(ops, cdt, tol, Hh, G, d, dv, rot):
    """One pass over projected rows with the half layout, amplified cosines and no norm, and the block means of the rows
    it writes -- as a launch of its own for many rows, inside the same launch for one row each -- against the chain
    of plain ops."""
    H, R = ops
    torch.manual_seed(d + dv)
    for lens, pos0 in (([37, 1, 20], [0, 9, 130]), ([1, 1, 1, 1], [15, 4, 31, 200]), ([1, 1], [5, 11]), ([2], [10])):
        md, npages, _ = meta_of(lens, pos0, DEV)
        T = sum(lens)
        z = torch.randn(T, (Hh + G) * d + G * dv + 5, device=DEV)
        kc, vc = torch.randn(npages, 16, G * d, device=DEV).to(cdt), torch.randn(npages, 16, G * dv, device=DEV).to(cdt)
        kc2, vc2 = kc.clone(), vc.clone()
        q1, q2 = torch.empty(T, Hh * d, device=DEV), torch.empty(T, Hh * d, device=DEV)
        b1 = blocks_of(lens, pos0, 6, 16, DEV, G * d, G * dv, cdt)
        b2 = (b1[0].clone(), b1[1].clone()) + b1[2:]
        kw = dict(rot=rot, norm=False, half=True)
        H.qkv_conv_rope_store(z, None, None, md, Hh, G, d, dv, q1, kc, vc, blocks=b1, **kw)
        R.qkv_conv_rope_store(z, None, None, md, Hh, G, d, dv, q2, kc2, vc2, blocks=b2, **kw)
        close(q1, q2, 2e-5)
        for x, y in ((kc, kc2), (vc, vc2), (b1[0], b2[0]), (b1[1], b2[1])):
            close(x, y, tol)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv", [(6, 2, 10, 14), (3, 1, 64, 64), (4, 2, 96, 96), (4, 4, 32, 32), (4, 2, 128, 128), (2, 1, 64, 128),
                                       (2, 2, 128, 64), (2, 1, 80, 48)])
def test_attention_over_a_window_and_pooled_blocks(ops, cdt, tol, Hh, G, d, dv):
    """Window tokens and earlier blocks in one softmax: prompts of several row tiles, portions, single rows, with head
    gates; windows and blocks that divide a page, each other, or nothing; block pools wider than the heads need."""
    H, R = ops
    torch.manual_seed(d + dv)
    for lens, pos0, window, P in (([300, 17, 140], [0, 0, 0], 50, 6), ([200, 30], [300, 17], 33, 16), ([3, 1, 1], [70, 5, 333], 9, 4),
                                  ([260], [0], 1, 1), ([150, 20], [0, 40], 2, 40), ([1, 1], [600, 2], 70, 3), ([130], [0], 500, 8)):
        md, npages, _ = meta_of(lens, pos0, DEV)
        T = sum(lens)
        kc, vc = torch.randn(npages, 16, G * d, device=DEV).to(cdt), torch.randn(npages, 16, G * dv, device=DEV).to(cdt)
        kp, vp, tab, _ = blocks_of(lens, pos0, P, 16, DEV, G * d + 8, G * dv + 16, cdt)
        q = torch.randn(T, Hh * d, device=DEV)
        if cdt == torch.bfloat16:
            q = q.to(cdt).float()
        gate = torch.randn(T, Hh + 3, device=DEV)[:, 1:1 + Hh]
        args = (q, kc, vc, md, Hh, G, d, dv, d ** -0.5 * 1.5, 0.0, None, None, 0, 16, cdt)
        kw = dict(window=window, blocks=(kp, vp, tab, P), head_gate=gate)
        close(H.attn_paged(*args, **kw), R.attn_paged(*args, **kw), tol)
        o = torch.empty(T, Hh * dv, device=DEV)
        close(H.attn_paged(*args, out=o, **kw), R.attn_paged(*args, **kw), tol)


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_decode_rows_over_many_blocks_split_their_keys(ops, cdt, tol):
    """Few rows over a long window and hundreds of blocks: the keys are cut into ranges whose first ones hold only
    blocks; the merge applies the head gates."""
    H, R = ops
    torch.manual_seed(2)
    Hh, G, d, dv, window, P = 4, 2, 40, 24, 700, 3
    md, npages, _ = meta_of([1, 1], [3000, 900], DEV)
    kc, vc = torch.randn(npages, 16, G * d, device=DEV).to(cdt), torch.randn(npages, 16, G * dv, device=DEV).to(cdt)
    blocks = blocks_of([1, 1], [3000, 900], P, 16, DEV, G * d, G * dv, cdt)
    q, gate = torch.randn(2, Hh * d, device=DEV), torch.randn(2, Hh, device=DEV)
    args = (q, kc, vc, md, Hh, G, d, dv, 0.3, 0.0, None, None, 0, 16, cdt)
    kw = dict(window=window, blocks=blocks, head_gate=gate)
    close(H.attn_paged(*args, **kw), R.attn_paged(*args, **kw), tol)
    with pytest.raises(ValueError):
        H.attn_paged(*args, window=0, blocks=blocks)
    with pytest.raises(ValueError):
        H.attn_paged(*args, window=window, sink=0.0, blocks=blocks)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("D", [1, 35, 96, 2048, 2300, 4096, 8200, 8196])
def test_residual_update_from_two_normed_branches(ops, cdt, tol, D):
    """All parts together and each left out; rows that are column blocks of a wider buffer (whose other columns stay);
    widths that fit the registers and wider ones; one-number and vector weights of the norm behind it."""
    H, R = ops
    torch.manual_seed(D)
    T = 7
    wide = torch.randn(T, 2 * D, device=DEV)
    a, b, f = (torch.randn(T, D, device=DEV) * s for s in (3.0, 0.2, 1.0))
    wa, wb, nw = (torch.randn(D, device=DEV) for _ in range(3))
    one = torch.tensor([0.7], device=DEV)
    for kw in (dict(branches=((a, wa), (b, wb)), coef=0.5, add=f), dict(branches=((a, wa), (b, wb)), coef=1.3),
               dict(branches=((a, wa), (b, wb)), coef=0.5, add=f, norm_w=nw), dict(add=f, keep=False, norm_w=one),
               dict(add=f, keep=False), dict(add=f, norm_w=one), dict(norm_w=nw)):
        x1, x2 = wide.clone(), wide.clone()
        h1 = H.residual_branches_(x1[:, :D], eps=1e-6, out_dtype=cdt, **kw)
        h2 = R.residual_branches_(x2[:, :D], eps=1e-6, out_dtype=cdt, **kw)
        close(x1, x2, 1e-5)
        assert torch.equal(x1[:, D:], wide[:, D:])
        if "norm_w" in kw:
            close(h1, h2, tol)
        else:
            assert h1 is None and h2 is None
    idx = torch.tensor([6, 0, 3], dtype=torch.int32, device=DEV)
    close(H.group_rmsnorm(wide[:, :D], one, 1, 1e-6, cdt, row_idx=idx), R.group_rmsnorm(wide[:, :D], one, 1, 1e-6, cdt, row_idx=idx), tol)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("M,N,K", [(5, 70, 33), (130, 192, 256), (300, 200, 454), (1600, 4200, 136), (8, 200, 512), (1, 33, 72)])
def test_squared_relu_in_the_epilogue(ops, cdt, tol, M, N, K):
    H, R = ops
    torch.manual_seed(M + N)
    a, w = torch.randn(M, K, device=DEV).to(cdt), torch.randn(N, K, device=DEV).to(cdt)
    b = torch.randn(N, device=DEV)
    close(H.matmul_nt(a, w, relu2=True, out_dtype=cdt), R.matmul_nt(a, w, relu2=True, out_dtype=cdt), tol)
    close(H.matmul_nt(a, w, b, relu2=True), R.matmul_nt(a, w, b, relu2=True), 2e-5)
    z = torch.randn(M, K + 3, device=DEV)[:, 1:1 + K]
    assert torch.equal(H.cast_rows(z, cdt), R.cast_rows(z, cdt)) and H.cast_rows(z, cdt).dtype == cdt
    z = torch.randn(M, 4 * K, device=DEV)
    assert torch.equal(H.cast_rows(z, cdt), z.to(cdt))


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("D", [1, 36, 35, 2048, 9000])
def test_side_by_side_rows(ops, cdt, tol, D):
    """Two norms of a row (with and without a second weight, with a row added first) and the residual update of two
    sublayers (plain, dense, experts with identities), on rows that are column slices of wider ones."""
    H, R = ops
    torch.manual_seed(D)
    T, E, Z, top = 7, 5, 8, 3
    wide = torch.randn(T, 2 * D, device=DEV)
    w1, w2 = torch.randn(D, device=DEV), torch.randn(D, device=DEV)
    for add in (False, True):
        for second in (w2, None):
            xa, xb = wide.clone(), wide.clone()
            a1, a2 = H.rmsnorm_pair(xa[:, :D], w1, second, 1e-5, cdt, add=xa[:, D:] if add else None)
            b1, b2 = R.rmsnorm_pair(xb[:, :D], w1, second, 1e-5, cdt, add=xb[:, D:] if add else None)
            close(a1, b1, tol)
            close(xa, xb, 1e-6)
            assert (a2 is None) == (b2 is None)
            if a2 is not None:
                close(a2, b2, tol)
    a, b = torch.randn(T, D, device=DEV), torch.randn(T, D, device=DEV)
    h, y = torch.randn(T, D, device=DEV).to(cdt), torch.randn(T * top, D, device=DEV)
    route = R.moe_route_softmax_grouped(torch.randn(T, Z, device=DEV) * 2, None, top, 4, 3, 1.3)
    assert bool((route.ids >= E).any()) and bool((route.ids < E).any())
    y[int(route.offs[E]):] = float("nan")                                   # (rows of identity experts are never made)
    for kw in ({}, {"b": b, "wb": w2}, {"wb": w2, "moe": (y, route, h, E)}):
        xa, xb = wide.clone(), wide.clone()
        H.parallel_update_(xa[:, :D], a, w1, **kw)
        kr = dict(kw, moe=(y.nan_to_num(), route, h, E)) if "moe" in kw else kw
        R.parallel_update_(xb[:, :D], a, w1, **kr)
        close(xa, xb, 1e-5)


# the rounding of group norms, step for step: rows whose values lie in one thread's four columns, so that nothing but them is summed.  The
# second square comes first, but in an update and norm in one pass of up to 1,024 columns; that pass multiplies scale and weight first, the two
# steps in turn the row and its scale
@pytest.mark.parametrize("D", [4, 1024, 1028, 4096, 8192])
@pytest.mark.parametrize("form", ["norm", "add", "next", "in turn"])
def test_group_norm_rounding(ops, D, form):
    H, _ = ops
    f32 = np.float32
    fma = lambda a, b, c: f32(np.longdouble(a) * np.longdouble(b) + np.longdouble(c))
    rng = np.random.default_rng(D)
    T, eps = 200, f32(1e-6)
    x, y = np.zeros((T, D), f32), np.zeros((T, D), f32)
    x[:, :4], y[:, :4] = rng.standard_normal((2, T, 4))
    w, w2 = rng.standard_normal((2, D)).astype(f32)
    x_first = form == "next" and D <= 1024

    def scale(v):                                  # 1 / rms of rows of four values
        sq = lambda i: (v[:, i] * v[:, i]).astype(f32)
        ss = fma(v[:, 1], v[:, 1], sq(0)) if x_first else fma(v[:, 0], v[:, 0], sq(1))
        ss = fma(v[:, 3], v[:, 3], fma(v[:, 2], v[:, 2], ss))
        return (f32(1) / np.sqrt(ss / f32(D) + eps))[:, None]
    dev = lambda a: torch.from_numpy(a.copy()).to(DEV)
    new = fma(y[:, :4] * scale(y[:, :4]), w[None, :4], x[:, :4])
    xd = dev(x)
    if form == "norm":
        assert np.array_equal(H.group_rmsnorm(dev(y), dev(w), 1, float(eps), torch.float32).cpu().numpy()[:, :4], y[:, :4] * scale(y[:, :4]) * w[:4])
        return
    if form == "add":
        H.add_group_rmsnorm_(xd, dev(y), dev(w), 1, float(eps))
    else:
        h = H.add_group_rmsnorm_next_(xd, dev(y), dev(w), dev(w2), 1, float(eps), torch.float32, in_turn=form == "in turn").cpu().numpy()[:, :4]
        assert np.array_equal(h, new * scale(new) * w2[:4] if form == "in turn" else new * (scale(new) * w2[:4]))
    assert np.array_equal(xd.cpu().numpy()[:, :4], new)


# a layer's last update with the next layer's norms in its pass: the bits of the two steps in turn, for widths about the pieces of 1,024 columns, the
# widest that rows in registers take, and widths and alignments that only the two steps serve
@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,pad", [(4, 0), (1020, 0), (1024, 4), (1028, 0), (2048, 0), (4100, 0), (8192, 0), (8196, 0), (35, 0), (64, 3)])
def test_update_with_the_next_norms(ops, cdt, D, pad):
    H, R = ops
    torch.manual_seed(D + pad)
    T, E, Z, top = 7, 5, 8, 3
    wide = torch.randn(T, 2 * (D + pad), device=DEV)
    w1, w2, n1, n2 = (torch.randn(D, device=DEV) for _ in range(4))
    a, b = torch.randn(T, D, device=DEV), torch.randn(T, D, device=DEV)
    h, y = torch.randn(T, D, device=DEV).to(cdt), torch.randn(T * top, D, device=DEV)
    route = R.moe_route_softmax_grouped(torch.randn(T, Z, device=DEV) * 2, None, top, 4, 3, 1.3)
    y[int(route.offs[E]):] = float("nan")                                   # (rows of identity experts are never made)
    for bb, wb, moe in ((None, None, None), (b, w2, None), (None, w2, (y, route, h, E))):
        for second, add in ((n2, False), (None, False), (n2, True)):
            xa, xb = wide.clone(), wide.clone()
            extra = lambda x: x[:, D + pad:2 * D + pad] if add else None
            g = H.parallel_update_norms_(xa[:, :D], a, w1, bb, wb, moe, n1, second, 1e-5, cdt, add=extra(xa))
            H.parallel_update_(xb[:, :D], a, w1, bb, wb, moe)
            want = H.rmsnorm_pair(xb[:, :D], n1, second, 1e-5, cdt, add=extra(xb))
            assert torch.equal(xa, xb) and torch.equal(g[0], want[0]) and (torch.equal(g[1], want[1]) if second is not None else g[1] is None)
    route = H.moe_route_corrected(torch.randn(T, E, device=DEV), torch.randn(E, device=DEV) * 0.1, top)
    y = torch.randn(T * top, D, device=DEV)
    for groups in (1, 2):
        if D % groups:
            continue
        xa, xb = wide.clone(), wide.clone()
        g = H.add_group_rmsnorm_moe_next_(xa[:, :D], y, route, w1, n1, groups, 1e-6, cdt)
        H.add_group_rmsnorm_moe_(xb[:, :D], y, route, w1, groups, 1e-6)
        assert torch.equal(xa, xb) and torch.equal(g, H.group_rmsnorm(xb[:, :D], n1, groups, 1e-6, cdt))
        g = H.add_group_rmsnorm_next_(xa[:, :D], a, w1, n1, groups, 1e-6, cdt, in_turn=True)
        H.add_group_rmsnorm_(xb[:, :D], a, w1, groups, 1e-6)
        assert torch.equal(xa, xb) and torch.equal(g, H.group_rmsnorm(xb[:, :D], n1, groups, 1e-6, cdt))


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("qr,r,dr,rot", [(9, 11, 8, 8), (1536, 512, 64, 64), (0, 40, 0, 0), (4, 12, 3, 2), (300, 1, 0, 0), (0, 512, 512, 64)])
def test_latent_rows(ops, cdt, tol, qr, r, dr, rot):
    """Both latents' norms, the rotated key part and the place in the pool, in one pass; other rows of the pool stay."""
    H, R = ops
    torch.manual_seed(qr + r)
    md, n_pages, _ = meta_of([5, 40, 1], [0, 7, 3000], DEV)
    T = 46
    z = torch.randn(T, qr + r + dr + 3, device=DEV)
    qn, kn = torch.randn(max(qr, 1), device=DEV), torch.randn(r, device=DEV)
    pa = torch.randn(n_pages * 16, r + dr, device=DEV).to(cdt)
    pb = pa.clone()
    args = (z, qr, r, dr, qn if qr else None, kn, 1e-5, (rot, 500.0) if rot else None)
    a, b = H.latent_rows(*args, pa, md, cdt), R.latent_rows(*args, pb, md, cdt)
    close(pa, pb, tol)
    assert (a is None) == (qr == 0)
    if qr:
        close(a, b, tol)


@pytest.mark.parametrize("heads,kv,d,dv", [(4, 2, 7, 9), (3, 3, 1, 1), (2, 1, 64, 64), (3, 3, 48, 130), (2, 2, 128, 128), (6, 2, 130, 20),
                                           (1, 1, 256, 300), (2, 1, 100, 512), (2, 2, 256, 128), (16, 8, 64, 64), (2, 2, 32, 32), (3, 1, 64, 256)])
def test_gated_delta_scan_carries_state(ops, heads, kv, d, dv):
    """The gated delta rule over unequal requests, some continuing from states in scattered slots: portions longer and shorter
    than a staged round, one row each (the fused form), strong and weak decays; outputs and states."""
    H, R = ops
    torch.manual_seed(heads + d)
    for lens, pos0 in (([33, 1, 7, 16], [0, 5, 12, 3]), ([1, 1, 1], [4, 0, 9]), ([50], [0]), ([2, 2], [0, 40])):
        md, _, n_slots = meta_of(lens, pos0, DEV)
        T = sum(lens)
        qkv = torch.randn(T, 2 * kv * d + heads * dv, device=DEV)
        zz = torch.randn(T, heads + 3, device=DEV)
        dec = torch.rand(T, heads * d, device=DEV) ** 3
        dec[:, ::5] = 1.0
        dec[:, 1::7] = 0.0
        gate, nw = torch.randn(T, heads * dv, device=DEV), 1 + 0.2 * torch.randn(dv, device=DEV)
        st = torch.randn(n_slots, heads, dv, d, device=DEV)
        for cdt, tol in ((torch.float32, 2e-4), (torch.bfloat16, 2e-2)):
            s1, s2 = st.clone(), st.clone()
            a = H.gated_delta_scan(qkv, zz[:, 2:2 + heads], dec, gate, nw, s1, md, heads, kv, d, dv, 1e-6, 1e-5, cdt)
            b = R.gated_delta_scan(qkv, zz[:, 2:2 + heads], dec, gate, nw, s2, md, heads, kv, d, dv, 1e-6, 1e-5, cdt)
            close(a, b, tol)
            close(s1, s2, 2e-4)                                             # (slots of nobody in the step stay as they were)


@pytest.mark.parametrize("T,E,top,groups,keep", [(50, 8, 2, 4, 3), (7, 12, 3, 4, 2), (300, 5, 2, 5, 3), (33, 6, 6, 2, 2), (20, 7, 1, 0, 0),
                                                 (64, 64, 8, 8, 4), (65, 64, 8, 8, 4), (9, 128, 16, 64, 9), (70, 150, 8, 10, 4), (3, 1024, 16, 32, 5),
                                                 (1, 3, 2, 3, 2), (500, 1024, 4, 0, 0)])
def test_corrected_softmax_routing_in_groups(ops, T, E, top, groups, keep):
    """Few tokens (one launch routes, counts and places) and many; corrections that make every choice score negative, none."""
    H, R = ops
    torch.manual_seed(T + E)
    logits = torch.randn(T, E + 3, device=DEV)[:, 1:1 + E] * 2
    for corr in (0.3 * torch.randn(E, device=DEV), 0.3 * torch.randn(E, device=DEV) - 3.0, None):
        a, b = (o.moe_route_softmax_grouped(logits, corr, top, groups, keep, 1.9) for o in (H, R))
        assert torch.equal(a.ids.cpu(), b.ids.cpu())
        close(a.w, b.w, 1e-5)
        assert torch.equal(a.offs.cpu(), b.offs.cpu())
        offs, dest = a.offs.cpu().long(), a.dest.cpu().long()
        assert bool(((dest >= offs[a.ids.cpu().long()]) & (dest < offs[a.ids.cpu().long() + 1])).all())
        assert torch.equal(a.rows.cpu().long()[dest], torch.arange(T)[:, None].expand(T, top))


@pytest.mark.parametrize("cdt,tol", DTYPES)
def test_clamped_gates_decays_and_bigram_rows(ops, cdt, tol):
    """The clamped gate product; a product whose epilogue turns it into decays (64- and 128-row tiles, few rows, an odd K);
    embedding rows with hashed bigrams (large multipliers, first tokens), one and two copies."""
    H, R = ops
    torch.manual_seed(3)
    gu = torch.randn(9, 2 * 300, device=DEV) * 4
    gu[0, :4] = torch.tensor([90.0, -90.0, 1.5, -1.5], device=DEV)
    for limit in (1.5, 1e4):
        close(H.gate_mul(gu, cdt, "clamped", limit=limit, alpha=1.702), R.gate_mul(gu, cdt, "clamped", limit=limit, alpha=1.702), tol)
    for M, N, K, n in ((5, 60, 33, 6), (3, 96, 64, 3), (150, 256, 24, 2), (70, 40, 16, 40)):
        a, w = torch.randn(M, K, device=DEV), (0.3 * torch.randn(N, K, device=DEV)).to(cdt)
        b, rates = torch.randn(N, device=DEV), torch.randn(n, device=DEV)
        close(H.matmul_nt(a, w, bias=b, decay=rates), R.matmul_nt(a, w, bias=b, decay=rates), tol)
    V, D, n = 40, 50, 23
    ids = torch.randint(0, V, (12,), dtype=torch.int32, device=DEV)
    prev = torch.randint(-1, V, (12,), dtype=torch.int32, device=DEV)
    prev[3] = -1
    tab, bt = torch.randn(V, D, device=DEV).to(cdt), torch.randn(n + 1, D, device=DEV).to(cdt)
    for mp, mc in ((7, 3), (1 << 30, (1 << 30) + 1), (0, 1)):
        for copies in (1, 2):
            close(H.embed_rows(ids, tab, copies=copies, bigram=(bt, prev, mp, mc)), R.embed_rows(ids, tab, copies=copies, bigram=(bt, prev, mp, mc)), 1e-6)


@pytest.mark.parametrize("cdt,tol", DTYPES)
@pytest.mark.parametrize("Hh,G,d,dv", [(3, 3, 14, 5), (4, 4, 128, 128), (6, 1, 64, 64), (5, 1, 576, 512), (32, 1, 512, 512), (7, 1, 256, 256), (3, 1, 128, 128),
                                       (40, 1, 128, 128)])
def test_attention_with_a_sink_per_head(ops, cdt, tol, Hh, G, d, dv):
    """A silent softmax entry of its own score in every head, loud and next to nothing, with head gates and windows, through
    every attention kernel: prompts, single rows over short contexts, single rows whose keys are cut into ranges, portions."""
    H, R = ops
    torch.manual_seed(Hh + d)
    sink = torch.randn(Hh, device=DEV) * 3
    sink[0] = -60.0
    for lens, pos0 in (([40, 150], [0, 33]), ([1, 1, 1], [0, 20, 900]), ([1], [1500]), ([2, 3], [500, 0])):
        md, n_pages, _ = meta_of(lens, pos0, DEV)
        kc = (torch.randn(n_pages, 16, G * d, device=DEV) * 0.3).to(cdt)
        vc = kc if G == 1 and dv <= d else (torch.randn(n_pages, 16, G * dv, device=DEV) * 0.3).to(cdt)
        q = torch.randn(sum(lens), Hh * d, device=DEV)
        hg = torch.randn(sum(lens), Hh + 2, device=DEV)[:, 1:1 + Hh]
        for window in (0, 50):
            for s, g in ((sink, hg), (sink, None), (None, hg)):
                kw = dict(scale=d ** -0.5, softcap=0.0, r1=None, r2=None, chunk=0, page_size=16, out_dtype=cdt, window=window, sink=s, head_gate=g)
                close(H.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), R.attn_paged(q, kc, vc, md, Hh, G, d, dv, **kw), tol)
