"""GPU parity of the recompute-selection kernels against the CPU oracle:
deviation keys bit-exact (fixed reduction order), selected indices bit-exact
(ties to the lower index), merge bit-exact."""
import numpy as np
import pytest
import torch

from daric_amd import cache_ops
from oracle import select as osel
from tests.gpu_util import make_layer, same_bytes, to_dev

pytestmark = pytest.mark.gpu


def setup_case(dev, layout="nhd", dtype=torch.bfloat16, nb=64, ps=16, h=4, d=64, L=2,
               chunk_tokens=(100, 64, 37), k_frac=0.15, seed=0):
    g = torch.Generator().manual_seed(seed)
    layers = [make_layer(layout, nb, ps, h, d, dtype, g) for _ in range(L)]
    pf = layers[0][1]
    perm = np.random.default_rng(seed).permutation(np.arange(1, nb)).tolist()
    bt, chunks, p, row = [], [], 0, 0
    for n in chunk_tokens:
        npg = -(-n // ps)
        chunks.append((len(bt), row, n, max(1, int(round(k_frac * n)))))
        bt.extend(perm[p:p + npg])
        p += npg
        row += n
    T = row
    bt = np.asarray(bt, np.int32)
    # recomputed K = cached K + heavy-tailed noise (config 3 style)
    kv = osel.k_rows_view(layers[0][0], pf)
    hh = kv.shape[2]
    rng = np.random.default_rng(seed + 1)
    k_new = torch.empty(L, T, hh, d if layout != "mla" else h * d, dtype=torch.bfloat16)
    v_new = torch.randn(L, T, hh, k_new.shape[3], generator=g).to(torch.bfloat16)
    for l, (t, _) in enumerate(layers):
        kvl = osel.k_rows_view(t, pf)
        for (bo, ro, n, _k) in chunks:
            blk, s = osel.chunk_slots(bt, bo, n, kvl.shape[1])
            base = kvl[torch.as_tensor(blk), torch.as_tensor(s)].float()
            noise = torch.from_numpy(0.1 * rng.standard_t(3, size=tuple(base.shape))).float()
            k_new[l, ro:ro + n] = (base + noise).to(torch.bfloat16)
    return layers, pf, bt, chunks, k_new, v_new


@pytest.mark.parametrize("layout", ["nhd", "hnd", "pf", "packed"])
def test_deviation_topk_merge_parity(dev, layout):
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, layout)
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    btd = torch.from_numpy(bt).to(dev)
    keys_o = osel.deviation(cpu, pf, bt, k_new, chunks)
    keys_g = cache_ops.kv_deviation(gpu, pf, btd, k_new.to(dev), chunks)
    torch.cuda.synchronize()
    kg = keys_g.cpu().numpy()
    assert np.array_equal(kg.view(np.uint32), keys_o.view(np.uint32)), \
        f"{int((kg != keys_o).sum())} keys differ"
    kmax = max(c[3] for c in chunks) + 3
    sel_o = osel.topk_per_chunk(keys_o, chunks, kmax)
    sel_g = cache_ops.topk_per_chunk(keys_g, chunks, kmax=kmax)
    torch.cuda.synchronize()
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    osel.merge_rows(cpu, pf, bt, k_new, v_new, chunks, sel_o)
    cache_ops.merge_rows(gpu, pf, btd, k_new.to(dev), v_new.to(dev), chunks, sel_g)
    torch.cuda.synchronize()
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


@pytest.mark.parametrize("layout", ["nhd", "hnd", "pf", "packed", "mla"])
@pytest.mark.parametrize("row_dtype", [torch.bfloat16, torch.float16])
def test_quantising_merge_parity(dev, layout, row_dtype):
    """bf16/fp16 recomputed rows merged into an fp8 (e4m3) cache: codes of
    x / scale[l, h] (K and V scales differ per layer and head), bit-exact
    against the oracle; every other byte of the cache unchanged."""
    layers, pf, bt, chunks, _k, _v = setup_case(dev, layout, dtype=torch.uint8, d=64, h=4, L=3)
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    kv = osel.k_rows_view(cpu[0], pf)
    L, H, D = len(cpu), kv.shape[2], kv.shape[3]
    T = chunks[-1][1] + chunks[-1][2]
    g = torch.Generator().manual_seed(21)
    k_new = (torch.randn(L, T, H, D, generator=g) * 5).to(row_dtype)
    v_new = (torch.randn(L, T, H, D, generator=g) * 5).to(row_dtype)
    k_new[0, 0, 0, :4] = torch.tensor([1e4, -1e4, 0.0, -0.0])        # saturation and signed zero
    k_new[0, 0, 0, 4:8] = torch.tensor([float("inf"), -float("inf"), 1e-39, 3e38]).to(row_dtype)
    k_new[0, 0, 0, 8:10] = torch.tensor([float("nan"), -float("nan")]).to(row_dtype)   # NaN codes keep the sign
    ks = (0.004 + 0.03 * torch.rand(L, H, generator=g)).float()
    vs = (0.004 + 0.03 * torch.rand(L, H, generator=g)).float()
    # scales outside [2^-60, 2^60] take the kernel's dividing path: rows scaled
    # alike keep bf16 codes in range (fp16 rows saturate or vanish)
    hv = min(1, H - 1)
    ks[1, 0] = 2.0 ** -70
    vs[2, hv] = 2.0 ** 62
    v_new[2, :, hv] = (v_new[2, :, hv].float() * 2.0 ** 62).to(row_dtype)
    kmax = max(c[3] for c in chunks)
    sel = np.full((L, len(chunks), kmax), -1, np.int32)
    rng = np.random.default_rng(5)
    for l in range(L):
        for c, (_bo, _ro, n, k) in enumerate(chunks):
            sel[l, c, :k] = np.sort(rng.choice(n, size=k, replace=False))
    sel[0, 0, 0] = 0
    osel.merge_rows(cpu, pf, bt, k_new, v_new, chunks, sel, k_scales=ks.numpy(), v_scales=vs.numpy())
    cache_ops.merge_rows(gpu, pf, torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev), chunks,
                         torch.from_numpy(sel).to(dev), k_scales=ks.to(dev), v_scales=vs.to(dev))
    torch.cuda.synchronize()
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


@pytest.mark.parametrize("h,d", [(8, 128), (4, 60)])
def test_merge_of_indices_in_any_slot(dev, h, d):
    """merge_rows takes a caller's own indices: a chunk's first min(k, kmax)
    slots may hold them in any place, also past as many slots as it has tokens
    (row kernel: batches of 8 slots; 120-byte rows: element kernel)."""
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", h=h, d=d, chunk_tokens=(3, 20, 1, 40))
    chunks = [c[:3] + (k,) for c, k in zip(chunks, (60, 33, 9, 17))]
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    sel = np.full((len(cpu), len(chunks), 60), -1, np.int32)
    for l in range(len(cpu)):
        sel[l, 0, [0, 30, 59]] = [2, 0, 1]
        sel[l, 1, [32, 5, 24]] = [19, 0, 7]
        sel[l, 2, 8] = 0
        sel[l, 3, :17] = np.arange(17)
    osel.merge_rows(cpu, pf, bt, k_new, v_new, chunks, sel)
    cache_ops.merge_rows(gpu, pf, torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev), chunks,
                         torch.from_numpy(sel).to(dev))
    torch.cuda.synchronize()
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


def test_quantising_merge_argument_errors(dev):
    layers, pf, bt, chunks, _k, _v = setup_case(dev, "nhd", dtype=torch.uint8, L=1)
    gpu = [to_dev(t, dev) for t, _ in layers]
    T = chunks[-1][1] + chunks[-1][2]
    k_new = torch.zeros(1, T, 4, 64, dtype=torch.bfloat16, device=dev)
    sel = torch.zeros(1, len(chunks), 1, dtype=torch.int32, device=dev)
    btd = torch.from_numpy(bt).to(dev)
    sc = torch.ones(1, 4, device=dev)
    with pytest.raises(RuntimeError, match="needs k_scales"):
        cache_ops.merge_rows(gpu, pf, btd, k_new, k_new, chunks, sel)
    with pytest.raises(RuntimeError, match="needs v_scales"):
        cache_ops.merge_rows(gpu, pf, btd, k_new, k_new, chunks, sel, k_scales=sc)
    with pytest.raises(RuntimeError, match="contiguous float32"):
        cache_ops.merge_rows(gpu, pf, btd, k_new, k_new, chunks, sel, k_scales=sc[:, :2], v_scales=sc)
    bf = [torch.zeros(2, 8, 16, 4, 64, dtype=torch.bfloat16, device=dev)]
    with pytest.raises(RuntimeError, match="element type"):
        cache_ops.merge_rows(bf, False, btd, k_new.half(), k_new.half(), chunks, sel)
    with pytest.raises(RuntimeError, match="apply only"):
        cache_ops.merge_rows(bf, False, btd, k_new, k_new, chunks, sel, k_scales=sc, v_scales=sc)


def test_topk_ties_and_edge_k(dev):
    rng = np.random.default_rng(7)
    L, T = 2, 3000
    keys = rng.integers(0, 4, (L, T)).astype(np.float32)    # massive ties
    keys[0, 17] = np.inf
    keys[1, 5] = np.array([0x7FC00000], np.uint32).view(np.float32)[0]
    chunks = [(0, 0, 512, 77), (0, 512, 2048, 205), (0, 2560, 400, 0), (0, 2960, 40, 40),
              (0, 2999, 1, 5)]
    kmax = 205
    want = osel.topk_per_chunk(keys, chunks, kmax)
    got = cache_ops.topk_per_chunk(torch.from_numpy(keys).to(dev), chunks, kmax=kmax)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)


def test_topk_random_distinct(dev):
    rng = np.random.default_rng(8)
    keys = rng.random((3, 8192)).astype(np.float32)
    chunks = [(0, 0, 8192, 1229), (0, 0, 100, 1)]
    want = osel.topk_per_chunk(keys, chunks, 1229)
    got = cache_ops.topk_per_chunk(torch.from_numpy(keys).to(dev), chunks, kmax=1229)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)


def topk_keys(kind, rng, n):
    if kind == "spread":
        return (rng.standard_t(3, n) ** 2).astype(np.float32)
    if kind == "few":                                  # ties at the k-th key
        return rng.integers(0, 3, n).astype(np.float32)
    if kind == "near":                                 # one exponent: the last bits decide
        return (np.float32(1.0) + rng.integers(0, 500, n).astype(np.float32) * np.float32(2.0 ** -23))
    return np.zeros(n, np.float32)                     # every key the same


# Chunk lengths at the edges of the top-k's workgroups (1, 4 and 16 wavefronts,
# 4, 8 and 32 keys per lane, keys from memory), each with small, half, nearly all
# and all tokens wanted, and more than there are.
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 8192, 8193, 32767, 32768, 32769])
@pytest.mark.parametrize("kind", ["spread", "few", "near", "zero"])
def test_topk_workgroup_edges(dev, n, kind):
    rng = np.random.default_rng(n)
    short = max(1, n // 3)
    keys = np.stack([topk_keys(kind, rng, n + short) for _ in range(2)])
    if kind == "spread" and n > 8:
        keys[0, n // 2] = np.inf
        keys[1, 3] = np.array([0x7FC00000], np.uint32).view(np.float32)[0]
    ks = sorted({1, 2, n // 2, n - 1, n, n + 3} - {0})
    chunks = [(0, 0, n, k) for k in ks] + [(0, n, short, max(1, short // 5)), (0, n, short, 0)]
    kmax = max(min(c[2], c[3]) for c in chunks) + 2
    want = osel.topk_per_chunk(keys, chunks, kmax)
    got = cache_ops.topk_per_chunk(torch.from_numpy(keys).to(dev), chunks, kmax=kmax)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)


# More chunks than CUs, where those of up to 8192 tokens take fewer lanes, and four
# times as many, where those of more than 32768 do; they share rows.
@pytest.mark.parametrize("n_chunks,longest", [(128, 4097), (129, 2049), (129, 4097), (129, 8192), (129, 8193),
                                              (512, 32769), (513, 32769), (513, 40001)])
def test_topk_of_many_long_chunks(dev, n_chunks, longest):
    rng = np.random.default_rng(longest)
    keys = np.stack([topk_keys(kind, rng, longest + n_chunks) for kind in ("spread", "few")])
    chunks = [(0, c, longest if c == 3 else int(rng.integers(1, longest + 1)), int(rng.integers(0, 400)))
              for c in range(n_chunks)]
    kmax = 401
    want = osel.topk_per_chunk(keys, chunks, kmax)
    got = cache_ops.topk_per_chunk(torch.from_numpy(keys).to(dev), chunks, kmax=kmax)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)


# A long chunk beside short ones at the edges of the forms that a part of its
# workgroup does.
@pytest.mark.parametrize("long", [257, 2049, 8192, 8193, 32769])
@pytest.mark.parametrize("kind", ["spread", "few", "zero"])
def test_topk_of_uneven_lengths(dev, long, kind):
    rng = np.random.default_rng(long)
    lens = [long, 1, 64, 256, 257, 0, 2047, 2048, 2049, 300]
    keys = np.stack([topk_keys(kind, rng, long + 300) for _ in range(3)])
    chunks = []
    for n in lens:
        n = min(n, long)
        chunks += [(0, long + 300 - n, n, k) for k in sorted({0, 1, n // 3, n, n + 2})]
    kmax = long + 1
    want = osel.topk_per_chunk(keys, chunks, kmax)
    got = cache_ops.topk_per_chunk(torch.from_numpy(keys).to(dev), chunks, kmax=kmax)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)


# Rows of 1, 8, 9, 16, 17, 32, 33 and 64 vectors of 8: the lanes that share a
# token in the deviation kernel, whole and partly filled.
@pytest.mark.parametrize("h,d", [(1, 8), (1, 64), (3, 24), (1, 128), (1, 136), (2, 128), (3, 88), (4, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.uint8])
def test_deviation_lane_groups(dev, h, d, dtype):
    layers, pf, bt, chunks, k_new, _v = setup_case(dev, "nhd", nb=60, h=h, d=d, L=2, dtype=dtype,
                                                   chunk_tokens=(133, 1, 70), seed=11)
    scales = None
    if dtype == torch.uint8:
        k_new = k_new.to(torch.bfloat16) if k_new.dtype == torch.uint8 else k_new
        scales = (0.5 + torch.rand(2, h, generator=torch.Generator().manual_seed(5))).float()
    want = osel.deviation([t for t, _ in layers], pf, bt, k_new, chunks,
                          **({} if scales is None else {"k_scales": scales.numpy()}))
    got = cache_ops.kv_deviation([to_dev(t, dev) for t, _ in layers], pf, torch.from_numpy(bt).to(dev),
                                 k_new.to(dev), chunks, k_scales=None if scales is None else scales.to(dev))
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy().view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("quant", [False, True])
def test_merge_of_uneven_counts(dev, quant):
    """Chunks that select none, one, a few and nearly all of their tokens: the
    row batches follow each chunk's own count, in merge_rows and select_merge."""
    dtype = torch.uint8 if quant else torch.bfloat16
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", nb=400, h=2, d=64, L=2, dtype=dtype,
                                                      chunk_tokens=(40, 2300, 17, 64, 900), seed=13)
    ks = (0, 2250, 17, 1, 130)
    chunks = [tuple(c[:3]) + (k,) + tuple(c[4:]) for c, k in zip(chunks, ks)]
    if k_new.dtype == torch.uint8:
        g = torch.Generator().manual_seed(3)
        k_new, v_new = (torch.randn(k_new.shape, generator=g).to(torch.bfloat16) for _ in range(2))
    sc = [torch.full((2, 2), 0.5 + 0.25 * i) for i in range(2)] if quant else [None, None]
    kw = dict(k_scales=sc[0].numpy(), v_scales=sc[1].numpy()) if quant else {}
    cpu = [t.clone() for t, _ in layers]
    keys = osel.deviation(cpu, pf, bt, k_new, chunks, **({"k_scales": sc[0].numpy()} if quant else {}))
    sel = osel.topk_per_chunk(np.asarray(keys, np.float32), chunks, max(ks))
    osel.merge_rows(cpu, pf, bt, k_new, v_new, chunks, sel, **kw)
    gpu = [to_dev(t, dev) for t, _ in layers]
    gk = dict(k_scales=sc[0].to(dev), v_scales=sc[1].to(dev)) if quant else {}
    _, got = cache_ops.select_merge(gpu, pf, torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev), chunks, **gk)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), sel)
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


def test_deviation_llama_shape(dev):
    # H*D = 1024 (two reduction rounds per lane), as benchmark configuration 3
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", nb=80, h=8, d=128, L=2,
                                                      chunk_tokens=(512, 512), seed=3)
    cpu = [t for t, _ in layers]
    keys_o = osel.deviation(cpu, pf, bt, k_new, chunks)
    keys_g = cache_ops.kv_deviation([to_dev(t, dev) for t in cpu], pf, torch.from_numpy(bt).to(dev),
                                    k_new.to(dev), chunks)
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))


@pytest.mark.parametrize("layout", ["nhd", "pf"])
def test_deviation_fp8_with_scales(dev, layout):
    """fp8 (e4m3) cache with per-(layer, head) scales: cached K is dequantised
    as float32(code * scale) before the fixed-order sum (configuration 5's
    selection on an fp8 cache). Keys and indices bit-exact."""
    from oracle import fp8 as ofp8
    g = torch.Generator().manual_seed(11)
    L, nb, ps, h, d = 2, 40, 16, 4, 64
    layers = [make_layer(layout, nb, ps, h, d, torch.uint8, g) for _ in range(L)]
    pf = layers[0][1]
    cpu = [t for t, _ in layers]
    scales = (torch.rand(L, h, generator=g) * 0.05 + 0.01).float()
    perm = np.random.default_rng(11).permutation(np.arange(1, nb)).tolist()
    chunk_tokens = (200, 97)
    bt, chunks, p, row = [], [], 0, 0
    for n in chunk_tokens:
        npg = -(-n // ps)
        chunks.append((len(bt), row, n, max(1, int(round(0.1 * n)))))
        bt.extend(perm[p:p + npg])
        p += npg
        row += n
    bt = np.asarray(bt, np.int32)
    T = row
    rng = np.random.default_rng(12)
    k_new = torch.empty(L, T, h, d, dtype=torch.bfloat16)
    for l in range(L):
        kv = osel.k_rows_view(cpu[l], pf)
        for (bo, ro, n, _k) in chunks:
            blk, s = osel.chunk_slots(bt, bo, n, ps)
            codes = kv[torch.as_tensor(blk), torch.as_tensor(s)].numpy()
            vals = ofp8.decode(codes) * scales[l].numpy()[:, None]
            noise = 0.01 * rng.standard_t(3, size=vals.shape)
            k_new[l, ro:ro + n] = torch.from_numpy((vals + noise).astype(np.float32)).to(torch.bfloat16)
    keys_o = osel.deviation(cpu, pf, bt, k_new, chunks, k_scales=scales.numpy())
    keys_g = cache_ops.kv_deviation([to_dev(t, dev) for t in cpu], pf, torch.from_numpy(bt).to(dev),
                                    k_new.to(dev), chunks, k_scales=scales.to(dev))
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    kmax = max(c[3] for c in chunks)
    sel_o = osel.topk_per_chunk(keys_o, chunks, kmax)
    sel_g = cache_ops.topk_per_chunk(keys_g, chunks, kmax=kmax)
    torch.cuda.synchronize()
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)


def test_deviation_allocated_keys_on_a_side_stream(dev):
    """kv_deviation allocating its own keys while launching on another stream:
    the zero fill is ordered before the kernel, so the rows outside every
    chunk read 0 and the chunk rows match the oracle."""
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", chunk_tokens=(100, 64, 37))
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    # leave rows 0..9 and the rows after the last chunk outside every chunk
    T = k_new.shape[1] + 24
    kn = torch.zeros(k_new.shape[0], T, *k_new.shape[2:], dtype=k_new.dtype)
    kn[:, 10:10 + k_new.shape[1]] = k_new
    moved = [(bo, ro + 10, n, k) for (bo, ro, n, k) in chunks]
    side = torch.cuda.Stream()
    btd, knd = torch.from_numpy(bt).to(dev), kn.to(dev)
    torch.cuda.synchronize()
    keys = cache_ops.kv_deviation(gpu, pf, btd, knd, moved, stream=side.cuda_stream)
    side.synchronize()
    want = osel.deviation(cpu, pf, bt, kn, moved)
    assert np.array_equal(keys.cpu().numpy().view(np.uint32), want.view(np.uint32))
    assert not keys[:, :10].any() and not keys[:, 10 + k_new.shape[1]:].any()


@pytest.mark.parametrize("moved", [
    lambda c: c,                                            # one after another over all rows: no fill
    lambda c: [c[2], c[0], c[1]],                           # all rows, another order
    lambda c: c[:2],                                        # rows after the last
    lambda c: c[1:],                                        # rows before the first
    lambda c: [c[0], c[2]],                                 # a gap
    lambda c: [c[0][:2] + (97,) + c[0][3:], c[1], c[2]],    # a gap of three rows
])
@pytest.mark.parametrize("one_call", [False, True])
def test_allocated_keys_cover_rows(dev, moved, one_call):
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", chunk_tokens=(100, 64, 37))
    chunks = moved(chunks)
    bt = bt.copy()
    bt[0] = 1 << 20             # a block id out of range: key 0, nothing read
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    btd, knd, vnd = torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev)
    want = osel.deviation(cpu, pf, bt, k_new, chunks)
    for _ in range(4):          # memory that held NaN before
        torch.full((len(gpu), k_new.shape[1]), float("nan"), device=dev)
    if one_call:
        keys, _ = cache_ops.select_merge(gpu, pf, btd, knd, vnd, chunks)
    else:
        keys = cache_ops.kv_deviation(gpu, pf, btd, knd, chunks)
    torch.cuda.synchronize()
    assert np.array_equal(keys.cpu().numpy().view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("n_long", [20000, 50000])
def test_topk_chunk_longer_than_lds_budget(dev, n_long):
    """A chunk of 20000 tokens, whose keys a workgroup of 1024 lanes holds in
    registers, or of 50000, whose keys are read from memory in every pass,
    beside a short one; indices bit-exact, ties to the lower index (the keys
    repeat every 97 tokens)."""
    rng = np.random.default_rng(11)
    n_short = 300
    base = rng.standard_normal(97).astype(np.float32) ** 2
    keys = np.concatenate([np.tile(base, n_long // 97 + 1)[:n_long],
                           rng.standard_normal(n_short).astype(np.float32) ** 2])[None, :].repeat(2, 0)
    keys[1] = keys[1][::-1]
    chunks = [(0, 0, n_long, 3001), (0, n_long, n_short, 45)]
    want = osel.topk_per_chunk(keys, chunks, 3001)
    got = cache_ops.topk_per_chunk(torch.from_numpy(keys.copy()).to(dev), chunks, kmax=3001)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)


def test_selection_over_more_than_65535_chunks(dev):
    """70000 chunks (past the 65535 a grid dimension holds): deviation, top-k
    and merge cut their grids into slices; keys, indices and merged bytes
    bit-exact against the oracle."""
    g = torch.Generator().manual_seed(13)
    n_chunks, ps, h, d = 70000, 1, 2, 64
    nb = n_chunks + 8
    layer = torch.randn(2, nb, ps, h, d, generator=g).to(torch.bfloat16)
    # one-token chunks, each on a page of its own: every merged slot is distinct
    bt = (torch.randperm(nb - 1, generator=g)[:n_chunks] + 1).numpy().astype(np.int32)
    chunks = [(c, c, 1, 1) for c in range(n_chunks)]
    k_new = torch.randn(1, n_chunks, h, d, generator=g).to(torch.bfloat16)
    v_new = torch.randn(1, n_chunks, h, d, generator=g).to(torch.bfloat16)
    gl = [layer.to(dev)]
    btd = torch.from_numpy(bt).to(dev)
    keys = cache_ops.kv_deviation(gl, False, btd, k_new.to(dev), chunks)
    sel = cache_ops.topk_per_chunk(keys, chunks, kmax=1)
    torch.cuda.synchronize()
    keys_o = osel.deviation([layer], False, bt, k_new, chunks)
    assert np.array_equal(keys.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    sel_o = osel.topk_per_chunk(keys_o, chunks, 1)
    assert np.array_equal(sel.cpu().numpy(), sel_o)
    cache_ops.merge_rows(gl, False, btd, k_new.to(dev), v_new.to(dev), chunks, sel)
    torch.cuda.synchronize()
    osel.merge_rows([layer], False, bt, k_new, v_new, chunks, sel_o)
    assert same_bytes(gl[0], layer)


def _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax, ks=None, vs=None):
    keys = osel.deviation(cpu, pf, bt, k_new, chunks, k_scales=ks)
    sel = osel.topk_per_chunk(keys, chunks, kmax)
    osel.merge_rows(cpu, pf, bt, k_new, v_new, chunks, sel, k_scales=ks, v_scales=vs)
    return keys, sel


@pytest.mark.parametrize("layout", ["nhd", "hnd", "pf", "packed", "mla"])
@pytest.mark.parametrize("mode", ["default", "keys_ready", "one_pass"])
def test_select_merge_matches_oracle(dev, layout, mode):
    """The whole selection in one call (the deviation kernel, then one
    workgroup per (layer, chunk) for top-k and merge; keys_ready: keys from an
    earlier kv_deviation; one_pass: those workgroups compute the keys too):
    keys, indices and merged bytes bit-exact against the oracle's three steps.
    Chunks start inside pages (tok_start) and one has k = 0."""
    keys_ready = mode == "keys_ready"
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, layout, chunk_tokens=(100, 64, 37, 300), seed=4)
    chunks = [c + (0,) for c in chunks]
    chunks[1] = (chunks[1][0], chunks[1][1], 50, chunks[1][3], 14)      # starts at token 14 of its pages
    chunks[2] = chunks[2][:3] + (0, 3)                                    # nothing selected
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    btd = torch.from_numpy(bt).to(dev)
    kmax = max(c[3] for c in chunks) + 2
    if layout == "mla":
        v_new = None
    keys_o, sel_o = _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax)
    keys = None
    if keys_ready:
        keys = cache_ops.kv_deviation(gpu, pf, btd, k_new.to(dev), chunks)
    keys_g, sel_g = cache_ops.select_merge(gpu, pf, btd, k_new.to(dev), None if v_new is None else v_new.to(dev),
                                           chunks, kmax=kmax, keys=keys, keys_ready=keys_ready,
                                           one_pass=mode == "one_pass")
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


@pytest.mark.parametrize("layout", ["nhd", "pf"])
def test_select_merge_head_dim_256(dev, layout):
    """256-wide heads (two per token: 1 KiB rows): select_merge against the
    oracle's three steps, bit-exact."""
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, layout, h=2, d=256, chunk_tokens=(100, 64, 37),
                                                      seed=37)
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    btd = torch.from_numpy(bt).to(dev)
    kmax = max(c[3] for c in chunks)
    keys_o, sel_o = _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax)
    keys_g, sel_g = cache_ops.select_merge(gpu, pf, btd, k_new.to(dev), v_new.to(dev), chunks, kmax=kmax)
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


@pytest.mark.parametrize("row_dtype,one_pass", [(torch.bfloat16, False), (torch.float16, False),
                                                (torch.bfloat16, True)])
def test_select_merge_fp8_cache(dev, row_dtype, one_pass):
    """fp8 (e4m3) cache: keys from cached K dequantised with the per-head K
    scales, rows quantised with the same K scales and the V scales."""
    layers, pf, bt, chunks, _k, _v = setup_case(dev, "nhd", dtype=torch.uint8, chunk_tokens=(100, 64, 37), L=2)
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    L, H, D = 2, 4, 64
    T = chunks[-1][1] + chunks[-1][2]
    g = torch.Generator().manual_seed(23)
    ks = (0.01 + 0.03 * torch.rand(L, H, generator=g)).float()
    vs = (0.01 + 0.03 * torch.rand(L, H, generator=g)).float()
    k_new = torch.randn(L, T, H, D, generator=g).to(row_dtype)
    v_new = torch.randn(L, T, H, D, generator=g).to(row_dtype)
    kmax = max(c[3] for c in chunks)
    keys_o, sel_o = _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax, ks.numpy(), vs.numpy())
    keys_g, sel_g = cache_ops.select_merge(gpu, pf, torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev),
                                           chunks, k_scales=ks.to(dev), v_scales=vs.to(dev), one_pass=one_pass)
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


def test_select_merge_long_chunk_takes_three_launches(dev):
    """A 9000-token chunk (past the 2048 keys whose top-k the fused kernel
    takes) beside a short one: the call runs deviation, top-k and merge in
    turn, with the same results."""
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", nb=600, h=2, d=64, L=1,
                                                      chunk_tokens=(9000, 120), seed=9)
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    kmax = max(c[3] for c in chunks)
    keys_o, sel_o = _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax)
    keys_g, sel_g = cache_ops.select_merge(gpu, pf, torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev),
                                           chunks)
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    assert same_bytes(gpu[0], cpu[0])


@pytest.mark.parametrize("mode", ["default", "keys_ready", "one_pass"])
@pytest.mark.parametrize("n", [2047, 2048, 2049])
def test_select_merge_at_the_fused_limit(dev, n, mode):
    """Chunks of 2048 tokens are the longest of the fused forms: one below, at
    and one past them, beside short chunks."""
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", nb=300, h=1, d=64, L=2, chunk_tokens=(n, 40, 500),
                                                      seed=n)
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    btd = torch.from_numpy(bt).to(dev)
    kmax = max(c[3] for c in chunks)
    keys_o, sel_o = _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax)
    keys = cache_ops.kv_deviation(gpu, pf, btd, k_new.to(dev), chunks) if mode == "keys_ready" else None
    keys_g, sel_g = cache_ops.select_merge(gpu, pf, btd, k_new.to(dev), v_new.to(dev), chunks, keys=keys,
                                           keys_ready=mode == "keys_ready", one_pass=mode == "one_pass")
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


@pytest.mark.parametrize("n_chunks,even", [(8, False), (60, False), (60, True), (100, False), (100, True)])
def test_select_merge_batch_tables(dev, n_chunks, even):
    """One chunk of 2100 tokens keeps the call from the fused form. The merge's
    batches of 8 chunks travel with the call's, of 60 in arguments of their own,
    of 100 in the ring; uneven counts, some 0, or two of every chunk."""
    rng = np.random.default_rng(n_chunks)
    lens = [2100] + [int(n) for n in rng.integers(8, 50, n_chunks - 1)]
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", nb=700, h=2, d=128, L=2, chunk_tokens=tuple(lens),
                                                      seed=n_chunks)
    ks = [2] * n_chunks if even else [int(rng.integers(0, min(n, 600) + 1)) * (i % 5 != 3) for i, n in enumerate(lens)]
    chunks = [c[:3] + (k,) for c, k in zip(chunks, ks)]
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    kmax = max(ks)
    keys_o, sel_o = _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax)
    keys_g, sel_g = cache_ops.select_merge(gpu, pf, torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev),
                                           chunks)
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)


@pytest.mark.parametrize("one_pass", [False, True])
def test_select_merge_many_selected_rows(dev, one_pass):
    """Chunks whose selected rows take more merge rounds than a fused
    workgroup handles well (Llama-3-8B rows, k = 154 of 1024): the call runs
    the three kernels, unless one_pass asks for the fused launch; results
    bit-exact either way."""
    layers, pf, bt, chunks, k_new, v_new = setup_case(dev, "nhd", nb=200, h=8, d=128, L=2,
                                                      chunk_tokens=(1024, 700), seed=5)
    cpu = [t for t, _ in layers]
    gpu = [to_dev(t, dev) for t in cpu]
    kmax = max(c[3] for c in chunks)
    keys_o, sel_o = _oracle_selection(cpu, pf, bt, k_new, v_new, chunks, kmax)
    keys_g, sel_g = cache_ops.select_merge(gpu, pf, torch.from_numpy(bt).to(dev), k_new.to(dev), v_new.to(dev),
                                           chunks, one_pass=one_pass)
    torch.cuda.synchronize()
    assert np.array_equal(keys_g.cpu().numpy().view(np.uint32), keys_o.view(np.uint32))
    assert np.array_equal(sel_g.cpu().numpy(), sel_o)
    for t, td in zip(cpu, gpu):
        assert same_bytes(td, t)
