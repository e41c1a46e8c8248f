"""Parity of the HIP kernels with the CPU oracle, through the C-ABI library.
Bar: bit-exact for indices, bytes and fp32 scores/means (the kernels reproduce
the reference's summation order, so scores are compared bit for bit as well;
the looser rel 1e-3 bound of the north star is implied)."""
import threading

import numpy as np
import pytest
import torch

import oracle as O
import synth
from golden.make_golden import select_inputs

pytestmark = pytest.mark.gpu

bits = lambda a: np.ascontiguousarray(a, np.float32).view(np.uint32)


def bf16_dev(bits_u16, dev):
    return torch.from_numpy(np.ascontiguousarray(bits_u16).view(np.int16)).to(dev).view(torch.bfloat16)


def i32(x, dev):
    return torch.tensor(np.asarray(x), dtype=torch.int32, device=dev)


def randn_bf16(dev, seed, shape):
    """Large caches are drawn on the device (seeded) and read back for the oracle."""
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    t = torch.randn(shape, device=dev, generator=g).to(torch.bfloat16)
    return t, t.view(torch.int16).cpu().numpy().view(np.uint16)


# ------------------------------------------------------------ block mean

@pytest.mark.parametrize("hkv,d,bs,n_layers", [(8, 128, 128, 2), (2, 64, 16, 1), (4, 128, 100, 3), (1, 8, 5, 1)])
def test_block_mean_matches_oracle(ucm, dev, hkv, d, bs, n_layers):
    from ucm_amd import ops

    nb, rows = 23, 40
    row = hkv * d
    caches_h = [synth.normal_bf16_bits(100 + l, (nb, bs, hkv, d)) for l in range(n_layers)]
    caches = [bf16_dev(c, dev) for c in caches_h]
    lp = ops.LayerPointers(caches)
    ids = synth.permutation(7, nb)[:15]
    slots = synth.permutation(8, rows)[:15]
    for mode in (ops.MEAN_F32, ops.MEAN_BF16_ROUND):
        repre = torch.full((n_layers, rows, row), 7.0, device=dev)
        ops.block_mean(lp, i32(ids, dev), i32(slots, dev), repre, bs, hkv, d, nb, mode=mode)
        got = repre.cpu().numpy()
        for l in range(n_layers):
            want = np.full((rows, row), 7.0, np.float32)
            O.block_mean_paged(caches_h[l], ids, slots, want, round_bf16=(mode == ops.MEAN_BF16_ROUND))
            assert np.array_equal(bits(got[l]), bits(want)), (mode, l)
    # the rounded mode is what torch's own mean in the model dtype stores, up to its summation order
    t = caches[0][torch.from_numpy(ids.astype(np.int64)).to(dev)].mean(1).float().reshape(len(ids), row)
    mine = repre[0][torch.from_numpy(slots.astype(np.int64)).to(dev)]
    assert torch.allclose(mine, t, rtol=2 ** -7, atol=1e-6)
    # MEAN_ABS: the same sums over the keys without their signs (the oracle on a cache whose sign bits are cleared)
    for mode in (ops.MEAN_F32, ops.MEAN_BF16_ROUND):
        repre = torch.full((n_layers, rows, row), 7.0, device=dev)
        ops.block_mean(lp, i32(ids, dev), i32(slots, dev), repre, bs, hkv, d, nb, mode=mode | ops.MEAN_ABS)
        got = repre.cpu().numpy()
        for l in range(n_layers):
            want = np.full((rows, row), 7.0, np.float32)
            O.block_mean_paged(caches_h[l] & np.uint16(0x7fff), ids, slots, want, round_bf16=(mode == ops.MEAN_BF16_ROUND))
            assert np.array_equal(bits(got[l]), bits(want)), (mode, l)
            assert (got[l][slots] >= 0).all()
    both = torch.zeros((n_layers, rows, row), dtype=torch.bfloat16, device=dev)
    ops.block_mean(lp, i32(ids, dev), i32(slots, dev), both, bs, hkv, d, nb, mode=ops.MEAN_ABS)   # a bf16 table of |k| means
    assert torch.equal(both[:, torch.from_numpy(slots.astype(np.int64)).to(dev)].float(),
                       repre[:, torch.from_numpy(slots.astype(np.int64)).to(dev)])


@pytest.mark.parametrize("hkv,d,bs", [(8, 128, 128), (2, 64, 16), (1, 8, 5)])
def test_block_mean_of_fp16_caches(ucm, dev, hkv, d, bs):
    """A model that runs in float16: the wrapper sees the cache's type, the kernel widens fp16 keys, and the rounding
    mode rounds to fp16 (the cache's type); a bf16 table from an fp16 cache is refused."""
    from ucm_amd import ops

    nb, rows, n_layers = 19, 30, 2
    row = hkv * d
    caches = [(torch.from_numpy(synth.normal_f32(130 + l, (nb, bs, hkv, d))) * 3).to(torch.float16).to(dev) for l in range(n_layers)]
    caches_h = [c.cpu().numpy().view(np.uint16) for c in caches]
    lp = ops.LayerPointers(caches)
    ids, slots = synth.permutation(9, nb)[:11], synth.permutation(10, rows)[:11]
    for mode in (ops.MEAN_F32, ops.MEAN_BF16_ROUND, ops.MEAN_F32 | ops.MEAN_ABS):
        repre = torch.full((n_layers, rows, row), 7.0, device=dev)
        ops.block_mean(lp, i32(ids, dev), i32(slots, dev), repre, bs, hkv, d, nb, mode=mode)
        got = repre.cpu().numpy()
        for l in range(n_layers):
            want = np.full((rows, row), 7.0, np.float32)
            keys = caches_h[l] & np.uint16(0x7fff) if mode & ops.MEAN_ABS else caches_h[l]
            O.block_mean_paged(keys, ids, slots, want, round_bf16=(mode == ops.MEAN_BF16_ROUND), keys_f16=True)
            assert np.array_equal(bits(got[l]), bits(want)), (mode, l)
    with pytest.raises(ops.UcmHipError):
        ops.block_mean(lp, i32(ids, dev), i32(slots, dev), torch.zeros((n_layers, rows, row), dtype=torch.bfloat16, device=dev),
                       bs, hkv, d, nb)


@pytest.mark.parametrize("hkv,d,bs,keys,table,mb,groups", [    # groups: what a persistent workgroup goes through, fits its LDS or more
    (8, 128, 16, "bfloat16", "bfloat16", 384, "fits"),     # two list entries side by side
    (8, 128, 32, "float16", "float32", 768, "more"),
    (8, 128, 16, "float16", "float32", 384, "short"),      # blocks of 16 tokens into an fp32 table: not persistent
    (8, 128, 128, "float16", "float32", 384, "fits"),
    (1, 8, 32, "bfloat16", "float32", 768, "more"),        # 256 entries side by side, several to a wave
    (1, 64, 32, "bfloat16", "float32", 768, "more"),
    (1, 64, 16, "bfloat16", "bfloat16", 384, "fits"),
    (1, 64, 32, "bfloat16", "bfloat16", 384, "fits"),
    (3, 96, 48, "bfloat16", "float32", 384, "more"),       # a row that does not divide the workgroup
    (16, 256, 16, "bfloat16", "bfloat16", 384, "fits"),    # two column groups
    (8, 128, 1024, "bfloat16", "bfloat16", 384, "few"),    # 192 groups are the least for persistent ones
])
def test_block_mean_of_large_launches(ucm, dev, hkv, d, bs, keys, table, mb, groups):
    """More than 256 MiB of keys (by repeated blocks) take persistent workgroups, which write their means out when they are done or,
    of more groups than LDS holds, on the way: every entry like the oracle's mean of its block, bad ids and slots skipped."""
    from ucm_amd import ops

    nb, L, row = 37 if bs < 1024 else 9, 3, hkv * d
    n = (mb << 20) // (L * bs * row * 2) + (333 if bs < 1024 else 33)
    threads = row // 8                                             # the launch as the host lays it out
    share = 256 // threads if threads < 256 and 256 % threads == 0 else 1
    total = L * (-(-n // share) if share > 1 else n * -(-threads // 256))
    kept = 158 * 1024 // ((32 if table == "float32" else 16) * 256 + 4 * max(share, 4))
    short = bs == 16 and table == "float32"
    assert groups == ("few" if total < 192 else "short" if short else "fits" if -(-total // 256) <= kept else "more")
    rows = n + 5
    f16 = keys == "float16"
    host = np.stack([synth.normal_f32(140 + l, (nb, bs, hkv, d)) for l in range(L)])
    caches = torch.from_numpy(host).to(torch.float16 if f16 else torch.bfloat16)
    caches_h = caches.view(torch.int16).numpy().view(np.uint16)
    caches = caches.to(dev)
    rng = np.random.default_rng(11)
    ids, slots = rng.integers(0, nb, n).astype(np.int32), rng.permutation(rows)[:n].astype(np.int32)
    bad = rng.permutation(n)[:9]
    good = np.ones(n, bool)
    good[bad] = False
    ids[bad[:5]] = [-1, nb, nb + 7, 2 ** 31 - 1, -2 ** 31]
    slots[bad[5:]] = [-1, rows, rows + 100, -2 ** 31]
    tdt = torch.float32 if table == "float32" else torch.bfloat16
    repre = torch.full((L, rows, row), 7.0, dtype=tdt, device=dev)
    ops.block_mean(ops.LayerPointers([caches[l] for l in range(L)]), i32(ids, dev), i32(slots, dev), repre, bs, hkv, d, nb,
                   mode=ops.MEAN_BF16_ROUND)
    for l in range(L):
        of_block = np.zeros((nb, row), np.float32)
        O.block_mean_paged(caches_h[l], np.arange(nb), np.arange(nb), of_block, round_bf16=True, keys_f16=f16)
        want = torch.full((rows, row), 7.0, dtype=tdt, device=dev)
        at = torch.from_numpy(slots[good].astype(np.int64)).to(dev)
        want[at] = torch.from_numpy(of_block).to(dev)[torch.from_numpy(ids[good].astype(np.int64)).to(dev)].to(tdt)
        assert torch.equal(repre[l], want), l


def test_block_mean_skips_bad_ids_and_layer_range(ucm, dev):
    from ucm_amd import ops

    hkv, d, bs, nb, rows = 8, 128, 128, 6, 9
    caches_h = [synth.normal_bf16_bits(200 + l, (nb, bs, hkv, d)) for l in range(3)]
    lp = ops.LayerPointers([bf16_dev(c, dev) for c in caches_h])
    repre = torch.zeros(3, rows, hkv * d, device=dev)
    ids = np.array([2, -1, 99, 5, 0], np.int32)
    slots = np.array([0, 1, 2, 100, 8], np.int32)
    ops.block_mean(lp, i32(ids, dev), i32(slots, dev), repre, bs, hkv, d, nb, first_layer=1, n_layers=1)
    got = repre.cpu().numpy()
    want = np.zeros((rows, hkv * d), np.float32)
    O.block_mean_paged(caches_h[1], [2, 0], [0, 8], want)
    assert np.array_equal(bits(got[1]), bits(want))
    assert not got[0].any() and not got[2].any()
    ops.block_mean(lp, i32([], dev), i32([], dev), repre, bs, hkv, d, nb)  # empty list is a no-op


# --------------------------------------------------------------- scoring

def run_select(ops, dev, q_np, repre_np, lens, topk, hkv, sw=1, ew=2, q_dtype=torch.float32, q_rows=None,
               block_tables=None, seq_lens=None, block_size=128, repre_dtype=torch.float32, tile=0, num_repre=1):
    """q_np [L, rows, Hq, D] fp32 values; repre_np [L, rows, Hkv*D] (values that
    repre_dtype holds exactly, so the oracle sees the same numbers).  Requests of up to 1024 blocks also go
    through the one-launch entry point, whose every output must equal the two launches'."""
    n_layers = repre_np.shape[0]
    lens = np.asarray(lens, np.int32)
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    q = torch.from_numpy(q_np).to(dev).to(q_dtype)
    repre = torch.from_numpy(repre_np).to(dev).to(repre_dtype)
    assert torch.equal(repre.float().cpu(), torch.from_numpy(repre_np))
    scores = torch.full((n_layers, repre_np.shape[1]), -123.0, device=dev)
    mx = int(lens.max(initial=0))
    ops.score_blocks(q, repre, i32(off, dev), i32(lens, dev), mx, hkv, scores,
                     q_rows=None if q_rows is None else i32(q_rows, dev), tile_blocks=tile, num_repre=num_repre)
    stride = max(mx, 1)
    idx = torch.full((n_layers, len(lens), stride), -1, dtype=torch.int32, device=dev)
    cnt = torch.full((n_layers, len(lens)), -1, dtype=torch.int32, device=dev)
    phys = sps = None
    bt = None
    if block_tables is not None:
        bt = i32(block_tables, dev)
        phys = torch.full_like(idx, -1)
    sl = None
    if seq_lens is not None:
        sl = i32(seq_lens, dev)
        sps = torch.full_like(cnt, -1)
    ops.topk_windows(scores, i32(off, dev), i32(lens, dev), i32(topk, dev), mx, idx, cnt, start_w=sw, end_w=ew,
                     block_tables=bt, phys_out=phys, seq_lens=sl, block_size=block_size, sparse_seq_lens=sps)
    torch.cuda.synchronize()
    out = dict(scores=scores.cpu().numpy(), idx=idx.cpu().numpy(), cnt=cnt.cpu().numpy(), off=off)
    if phys is not None:
        out["phys"] = phys.cpu().numpy()
    if sps is not None:
        out["sparse_seq_lens"] = sps.cpu().numpy()
    if mx <= 1024:
        fused = dict(scores=torch.full_like(scores, -123.0), idx=torch.full_like(idx, -1), cnt=torch.full_like(cnt, -1),
                     phys=None if phys is None else torch.full_like(phys, -1), sps=None if sps is None else torch.full_like(sps, -1))
        tickets = torch.zeros_like(cnt)
        # twice: the tickets must come back to zero; the second time with a total that understates the batch, so
        # that the grid is short and workgroups go on to a second and third tile
        for total in (0, max(int(lens.sum()) // 3, 1)):
            ops.score_select(q, repre, i32(off, dev), i32(lens, dev), i32(topk, dev), mx, hkv, fused["scores"], fused["idx"],
                             fused["cnt"], tickets, start_w=sw, end_w=ew, q_rows=None if q_rows is None else i32(q_rows, dev),
                             block_tables=bt, phys_out=fused["phys"], seq_lens=sl, block_size=block_size,
                             sparse_seq_lens=fused["sps"], tile_blocks=tile, total_blocks=total, num_repre=num_repre)
            torch.cuda.synchronize()
            assert not tickets.any(), "tickets left non-zero"
        assert torch.equal(fused["scores"].view(torch.int32), scores.view(torch.int32)), "fused scores differ"
        assert torch.equal(fused["cnt"], cnt), "fused counts differ"
        assert torch.equal(fused["idx"], idx), "fused selection differs"
        if phys is not None:
            assert torch.equal(fused["phys"], phys), "fused block-table lookup differs"
        if sps is not None:
            assert torch.equal(fused["sps"], sps), "fused sparse lengths differ"
    return out


def check_against_oracle(out, q_np, repre_np, lens, topk, hkv, sw=1, ew=2, q_rows=None, num_repre=1):
    n_layers = repre_np.shape[0]
    for l in range(n_layers):
        ql = q_np[l] if q_rows is None else q_np[l][np.asarray(q_rows)]
        widx, wcnt, wscores = O.select_topk_bs(ql[: len(lens)], repre_np[l], out["off"], lens, topk, hkv, num_krepre=num_repre,
                                               start_w=sw, end_w=ew, out_stride=out["idx"].shape[2] + sw + ew + max(topk))
        for r, n in enumerate(lens):
            a, b = out["off"][r], out["off"][r] + n
            if topk[r] > 0:  # the reference (and the oracle) skip scoring when k == 0
                assert np.array_equal(bits(out["scores"][l, a:b]), bits(wscores[a:b])), (l, r)
                assert out["cnt"][l, r] == wcnt[r], (l, r)
                assert np.array_equal(out["idx"][l, r, : wcnt[r]], widx[r, : wcnt[r]]), (l, r)


def test_golden_select_cases_on_gpu(ucm, dev, golden):
    from ucm_amd import ops

    z, meta = golden
    for name, seed, n, hq, hkv, d, k, sw, ew, b16 in meta["select"]:
        if d not in (64, 128):
            continue  # head sizes the kernel is not built for are refused (test_abi)
        q, repre = select_inputs(seed, n, hq, hkv, d, b16)
        out = run_select(ops, dev, q[None, None], repre.reshape(1, n, hkv * d), [n], [k], hkv, sw, ew)
        assert np.array_equal(bits(out["scores"][0, :n]), bits(z[f"select/{name}/scores"])), name
        want = z[f"select/{name}/idx"]
        assert out["cnt"][0, 0] == len(want), name
        assert np.array_equal(out["idx"][0, 0, : len(want)], want), name


@pytest.mark.parametrize("hkv,g,d", [(8, 4, 128), (8, 8, 128), (1, 8, 128), (2, 2, 64), (4, 1, 64), (16, 2, 128),
                                     (8, 4, 32), (2, 4, 96), (4, 2, 192), (8, 2, 256), (1, 16, 256)])
@pytest.mark.parametrize("q_dtype", [torch.float32, torch.bfloat16])
def test_ragged_batch_scores_and_selection(ucm, dev, hkv, g, d, q_dtype):
    from ucm_amd import ops

    n_layers = 3
    lens = [1, 2, 3, 4, 0, 17, 64, 65, 130, 33, 257]
    topk = [O.compute_topk_len(n) if n > 40 else max(n // 2, 1) for n in lens]
    rows = int(np.sum(lens))
    q = synth.normal_bf16_as_f32(31, (n_layers, len(lens), hkv * g, d))
    repre = synth.normal_f32(32, (n_layers, rows, hkv * d)) * np.float32(0.3)
    out = run_select(ops, dev, q, repre, lens, topk, hkv, q_dtype=q_dtype)
    check_against_oracle(out, q, repre, lens, topk, hkv)
    assert out["cnt"][0, 4] == 0  # the empty request selects nothing


@pytest.mark.parametrize("hkv,g,d,num_repre", [(8, 4, 128, 2), (4, 8, 128, 2), (2, 2, 64, 4), (1, 8, 128, 2), (4, 2, 64, 4)])
@pytest.mark.parametrize("q_dtype,repre_dtype", [(torch.float32, torch.float32), (torch.float16, torch.float32),
                                                 (torch.bfloat16, torch.bfloat16), (torch.float16, torch.bfloat16)])
def test_several_representatives_per_head_and_fp16_queries(ucm, dev, hkv, g, d, num_repre, q_dtype, repre_dtype):
    """numKrepre > 1: a block's score takes, per kv head, the largest of the dots with that head's representatives
    (k_repre rows laid out [kv head][representative][channel], cal_kpre_and_topk.cpp's kRepre); queries in any of the
    three types the model may run in, widened exactly."""
    from ucm_amd import ops

    lens = [3, 40, 0, 65, 130, 257]
    topk = [max(n // 3, 1) for n in lens]
    rows = int(np.sum(lens))
    q = synth.normal_bf16_as_f32(41, (2, len(lens), hkv * g, d))
    if q_dtype == torch.float16:
        q = torch.from_numpy(q).to(torch.float16).float().numpy()        # values fp16 holds exactly
    repre = synth.normal_f32(42, (2, rows, hkv * num_repre * d)) * np.float32(0.3)
    if repre_dtype == torch.bfloat16:
        repre = torch.from_numpy(repre).to(torch.bfloat16).float().numpy()
    out = run_select(ops, dev, q, repre, lens, topk, hkv, q_dtype=q_dtype, repre_dtype=repre_dtype, num_repre=num_repre)
    check_against_oracle(out, q, repre, lens, topk, hkv, num_repre=num_repre)


def as_bf16_values(a):
    """fp32 array rounded to the nearest bf16 value (torch's rounding, ties to even)."""
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(torch.bfloat16).float().numpy()


@pytest.mark.parametrize("hkv,g,d", [(8, 4, 128), (8, 8, 128), (1, 8, 128), (2, 2, 64), (4, 1, 64), (16, 2, 128),
                                     (8, 4, 32), (2, 4, 96), (4, 2, 192), (8, 2, 256), (1, 16, 256)])
@pytest.mark.parametrize("q_dtype", [torch.float32, torch.bfloat16])
def test_bf16_table_scores_like_the_widened_table(ucm, dev, hkv, g, d, q_dtype):
    """A bf16 representative table holds what the live path stores (ucm/sparse/gsa/gsa.py:640-652);
    scores and selections must equal the oracle's on the same values widened to fp32, bit for bit."""
    from ucm_amd import ops

    n_layers = 2
    lens = [1, 2, 3, 0, 17, 31, 32, 33, 64, 65, 130, 257]
    topk = [O.compute_topk_len(n) if n > 40 else max(n // 2, 1) for n in lens]
    rows = int(np.sum(lens))
    q = synth.normal_bf16_as_f32(33, (n_layers, len(lens), hkv * g, d))
    repre = as_bf16_values(synth.normal_f32(34, (n_layers, rows, hkv * d)) * np.float32(0.3))
    for tile in (5, 32):
        out = run_select(ops, dev, q, repre, lens, topk, hkv, q_dtype=q_dtype, repre_dtype=torch.bfloat16, tile=tile)
        check_against_oracle(out, q, repre, lens, topk, hkv)


@pytest.mark.parametrize("hkv,g,d,repre_dtype", [(8, 4, 128, torch.bfloat16), (2, 8, 64, torch.float32)])
def test_score_scale_gives_the_torch_variants_values(ucm, dev, hkv, g, d, repre_dtype):
    """scale = 1/kv_heads turns the score into the mean over ALL q heads of q[h] . k[kv head of h], what the
    reference's torch variant ranks by (TopkCal.cal_topk, ucm/sparse/gsa/gsa.py:386-412, one representative per
    block); scale = 1 leaves the bits of the unscaled call."""
    from ucm_amd import ops

    n_layers, lens = 2, np.array([37, 0, 130, 5], np.int32)
    rows, hq = int(lens.sum()), hkv * g
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    q = torch.from_numpy(synth.normal_f32(4100, (n_layers, len(lens), hq, d))).to(dev)
    repre = torch.from_numpy(synth.normal_f32(4101, (n_layers, rows, hkv * d))).to(dev).to(repre_dtype)
    plain, one, scaled = (torch.full((n_layers, rows), -5.0, device=dev) for _ in range(3))
    args = (q, repre, i32(off, dev), i32(lens, dev), int(lens.max()), hkv)
    ops.score_blocks(*args, plain)
    ops.score_blocks(*args, one, scale=1.0)
    ops.score_blocks(*args, scaled, scale=1.0 / hkv)
    assert torch.equal(plain, one)
    assert torch.equal(scaled, plain * np.float32(1.0 / hkv))          # one fp32 multiplication of the same score
    # the torch variant's formula, in fp64: expand every kv head to its g query heads, dot, mean over the q heads
    k = repre.double().view(n_layers, rows, hkv, 1, d).expand(-1, -1, -1, g, -1).reshape(n_layers, rows, hq, d)
    for r, (a, n) in enumerate(zip(off, lens)):
        want = torch.einsum("lhd,lbhd->lhb", q[:, r].double(), k[:, a : a + n]).mean(dim=1)
        assert torch.allclose(scaled[:, a : a + n].double(), want, rtol=1e-5, atol=1e-5), r


def test_bf16_table_from_the_paged_cache(ucm, dev):
    """keys -> bf16 means -> scores, against the oracle's rounded means; the bf16 table is the
    fp32 table of UCM_MEAN_BF16_ROUND with the low halves dropped."""
    from ucm_amd import ops

    hq, hkv, d, bs, nb, n_layers = 32, 8, 128, 128, 70, 2
    caches_h = [synth.normal_bf16_bits(81 + l, (nb, bs, hkv, d)) for l in range(n_layers)]
    lp = ops.LayerPointers([bf16_dev(c, dev) for c in caches_h])
    table = synth.permutation(83, nb)[:67]
    n = len(table)
    slots = np.arange(n)
    t16 = torch.full((n_layers, n + 2, hkv * d), 3.0, device=dev, dtype=torch.bfloat16)
    t32 = torch.full((n_layers, n + 2, hkv * d), 3.0, device=dev)
    ops.block_mean(lp, i32(table, dev), i32(slots, dev), t16, bs, hkv, d, nb)
    ops.block_mean(lp, i32(table, dev), i32(slots, dev), t32, bs, hkv, d, nb, mode=ops.MEAN_BF16_ROUND)
    assert torch.equal(t16.float(), t32)
    want = np.full((n_layers, n + 2, hkv * d), 3.0, np.float32)
    for l in range(n_layers):
        O.block_mean_paged(caches_h[l], table, slots, want[l], round_bf16=True)
    assert np.array_equal(bits(t16.float().cpu().numpy()), bits(want))
    with pytest.raises(ValueError):
        ops.block_mean(lp, i32(table, dev), i32(slots, dev), t32, bs, hkv, d, nb, mode=ops.MEAN_BF16_STORE)
    q = synth.normal_bf16_as_f32(84, (n_layers, 1, hq, d))
    out = run_select(ops, dev, q, want[:, :n], [n], [24], hkv, q_dtype=torch.bfloat16, repre_dtype=torch.bfloat16)
    check_against_oracle(out, q, want[:, :n], [n], [24], hkv)


def test_q_rows_indirection_and_tile_sizes(ucm, dev):
    from ucm_amd import ops

    hkv, g, d = 8, 4, 128
    lens = [70, 200, 9]
    topk = [19, 40, 5]
    q = synth.normal_bf16_as_f32(41, (2, 12, hkv * g, d))     # 12 token rows, requests read rows 11, 0, 5
    repre = synth.normal_f32(42, (2, int(np.sum(lens)), hkv * d))
    rows = [11, 0, 5]
    for tile in (1, 2, 7, 32, 4096):
        out = run_select(ops, dev, q, repre, lens, topk, hkv, q_dtype=torch.bfloat16, q_rows=rows, tile=tile)
        check_against_oracle(out, q, repre, lens, topk, hkv, q_rows=rows)


@pytest.mark.parametrize("repre_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tile", [2047, 2048, 2049, 4096])
def test_tiles_around_what_a_workgroup_holds(ucm, dev, tile, repre_dtype):
    """Requests of one and of several tiles at the largest tile a workgroup's scores have room for, and above it."""
    from ucm_amd import ops

    hkv, g, d, lens = 1, 2, 32, [2047, 2048, 2049, 4096, 5000, 1]
    off, rows = np.concatenate([[0], np.cumsum(lens)[:-1]]), int(np.sum(lens))
    q = synth.normal_bf16_as_f32(43, (len(lens), hkv * g, d))
    repre = as_bf16_values(synth.normal_f32(44, (rows, hkv * d)))
    scores = torch.zeros((1, rows), device=dev)
    ops.score_blocks(torch.from_numpy(q).to(dev)[None], torch.from_numpy(repre).to(dev).to(repre_dtype)[None], i32(off, dev), i32(lens, dev),
                     max(lens), hkv, scores, tile_blocks=tile)
    for r, n in enumerate(lens):
        want = O.kq_scores(O.q_head_mean(q[r], hkv), repre[off[r] : off[r] + n].reshape(n, hkv, 1, d))
        assert np.array_equal(bits(scores[0, off[r] : off[r] + n].cpu().numpy()), bits(want)), r


@pytest.mark.parametrize("repre_dtype", [torch.float32, torch.bfloat16])
def test_query_rows_outside_the_layer_are_skipped(ucm, dev, repre_dtype):
    """q_rows comes from device memory: a request whose query row is negative or past the layer's block of
    queries is not followed - its scores stay as they were - and the other requests are scored as usual."""
    from ucm_amd import ops

    hkv, g, d, n_tok = 8, 4, 128, 9
    lens = np.array([20, 70, 5, 33], np.int32)
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    rows = int(lens.sum())
    q = synth.normal_bf16_as_f32(61, (2, n_tok, hkv * g, d))
    repre = synth.bf16_widen(synth.bf16_round_bits(synth.normal_f32(62, (2, rows, hkv * d))))
    q_rows = np.array([3, n_tok, 8, -1], np.int32)          # the second is one past the end, the last negative
    scores = torch.full((2, rows), -5.0, device=dev)
    ops.score_blocks(torch.from_numpy(q).to(dev).to(torch.bfloat16), torch.from_numpy(repre).to(dev).to(repre_dtype),
                     i32(off, dev), i32(lens, dev), int(lens.max()), hkv, scores, q_rows=i32(q_rows, dev))
    got = scores.cpu().numpy()
    topk = np.full(len(lens), 4, np.int32)
    for l in range(2):
        ql = q[l][np.clip(q_rows, 0, n_tok - 1)]
        _, _, want = O.select_topk_bs(ql, repre[l], off, lens, topk, hkv)
        for r, ok in enumerate([True, False, True, False]):
            seg = slice(off[r], off[r] + lens[r])
            if ok:
                assert np.array_equal(bits(got[l][seg]), bits(want[seg])), (l, r)
            else:
                assert np.all(got[l][seg] == -5.0), (l, r)


@pytest.mark.parametrize("repre_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tile", [16, 64])
def test_fused_selection_of_whole_split_and_unfollowed_requests(ucm, dev, repre_dtype, tile):
    """The one-launch call selects from LDS when a workgroup holds the whole request, from memory otherwise; a request
    whose query row is out of range keeps the scores it had and is selected from them, as the two calls do."""
    from ucm_amd import ops

    hkv, g, d, n_tok = 8, 4, 128, 6
    lens = np.array([1, 15, 16, 17, 63, 64, 65, 130, 16, 70], np.int32)
    q_rows = np.array([0, 1, 2, 3, 4, 5, 0, 1, n_tok, -1], np.int32)        # the last two are not followed
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    topk = np.array([1, 6, 5, 7, 19, 64, 20, 9, 5, 8], np.int32)
    rows, mx = int(lens.sum()), int(lens.max())
    q = torch.from_numpy(synth.normal_bf16_as_f32(71, (2, n_tok, hkv * g, d))).to(dev).to(torch.bfloat16)
    repre = torch.from_numpy(synth.normal_f32(72, (2, rows, hkv * d))).to(dev).to(repre_dtype)
    old = torch.from_numpy(synth.normal_f32(73, (2, rows))).to(dev)
    args = (i32(off, dev), i32(lens, dev))
    out = []
    for fused in (False, True):
        scores, idx = old.clone(), torch.full((2, len(lens), mx), -1, dtype=torch.int32, device=dev)
        cnt, tickets = torch.full((2, len(lens)), -1, dtype=torch.int32, device=dev), torch.zeros((2, len(lens)), dtype=torch.int32, device=dev)
        if fused:
            ops.score_select(q, repre, *args, i32(topk, dev), mx, hkv, scores, idx, cnt, tickets, q_rows=i32(q_rows, dev), tile_blocks=tile)
            assert not tickets.any()
        else:
            ops.score_blocks(q, repre, *args, mx, hkv, scores, q_rows=i32(q_rows, dev), tile_blocks=tile)
            ops.topk_windows(scores, *args, i32(topk, dev), mx, idx, cnt)
        out.append((scores, idx, cnt))
    for a, b in zip(*out):
        assert torch.equal(a, b)
    assert torch.equal(out[1][0][:, off[8]:], old[:, off[8]:])


def test_many_requests_dense_tile_lookup(ucm, dev):
    """More requests than one wavefront scans at once (the tile -> request lookup runs in trips of 64),
    with empty requests in between, and the grid sized from the host-known total."""
    from ucm_amd import ops

    hkv, g, d = 4, 2, 64
    lens = synth.ints(45, 150, 0, 40).astype(np.int32)
    lens[[0, 63, 64, 65, 149]] = [0, 33, 0, 1, 40]
    topk = np.maximum(lens // 3, 1).astype(np.int32)
    rows = int(lens.sum())
    q = synth.normal_bf16_as_f32(46, (2, len(lens), hkv * g, d))
    repre = synth.normal_f32(47, (2, rows, hkv * d))
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    for tile in (3, 32):
        for total in (0, rows):
            scores = torch.full((2, rows), -5.0, device=dev)
            ops.score_blocks(torch.from_numpy(q).to(dev), torch.from_numpy(repre).to(dev), i32(off, dev),
                             i32(lens, dev), int(lens.max()), hkv, scores, total_blocks=total, tile_blocks=tile)
            got = scores.cpu().numpy()
            for l in range(2):
                _, _, want = O.select_topk_bs(q[l], repre[l], off, lens, topk, hkv)
                live = np.concatenate([np.arange(off[r], off[r] + lens[r]) for r in range(len(lens))])
                assert np.array_equal(bits(got[l][live]), bits(want[live])), (tile, total, l)


def test_config1_single_request_32k(ucm, dev):
    """Llama-3-8B shape, 32768 tokens = 256 blocks, top-16 + first 1 + last 2, keys -> means -> scores."""
    from ucm_amd import ops

    hq, hkv, d, bs, n = 32, 8, 128, 128, 256
    cache_d, cache_h = randn_bf16(dev, 51, (n, bs, hkv, d))
    lp = ops.LayerPointers([cache_d])
    table = synth.permutation(52, n)
    repre = torch.zeros(1, n, hkv * d, device=dev)
    ops.block_mean(lp, i32(table, dev), i32(np.arange(n), dev), repre, bs, hkv, d, n)
    want_repre = np.zeros((n, hkv * d), np.float32)
    O.block_mean_paged(cache_h, table, np.arange(n), want_repre)
    assert np.array_equal(bits(repre[0].cpu().numpy()), bits(want_repre))
    q = synth.normal_bf16_as_f32(53, (1, 1, hq, d))
    out = run_select(ops, dev, q, want_repre[None], [n], [19], hkv, block_tables=table[None], seq_lens=[n * bs])
    check_against_oracle(out, q, want_repre[None], [n], [19], hkv)
    sel = out["idx"][0, 0, :19]
    assert sel[0] == 0 and list(sel[-2:]) == [n - 2, n - 1]
    assert np.array_equal(out["phys"][0, 0, :19], table[sel])
    assert out["sparse_seq_lens"][0, 0] == 19 * bs
    # independent fp64 bound on the scores (rel 1e-3 of the north star)
    qm = q[0, 0].reshape(hkv, 4, d).astype(np.float64).mean(1)
    ref64 = np.einsum("hd,nhd->n", qm, want_repre.reshape(n, hkv, d).astype(np.float64))
    assert np.allclose(out["scores"][0, :n], ref64, rtol=1e-3, atol=1e-5)


def test_config4_shape_long_context_g8(ucm, dev):
    """Qwen2-72B shape: 64 query heads, g = 8, up to 1024 blocks, k = 2 % + windows."""
    from ucm_amd import ops

    hkv, g, d = 8, 8, 128
    lens = [1024, 512, 777]
    topk = [max(16, int(0.02 * n)) + 3 for n in lens]
    q = synth.normal_bf16_as_f32(61, (2, len(lens), hkv * g, d))
    repre = synth.normal_f32(62, (2, int(np.sum(lens)), hkv * d)) * np.float32(0.2)
    out = run_select(ops, dev, q, repre, lens, topk, hkv, q_dtype=torch.bfloat16)
    check_against_oracle(out, q, repre, lens, topk, hkv)


def test_incremental_repre_update(ucm, dev):
    """Decode-time update: only the newly filled block is reduced (ucm/sparse/gsa/gsa.py:234-236);
    every other row of the table must stay untouched."""
    from ucm_amd import ops

    hkv, d, bs, nb = 8, 128, 128, 12
    cache_h = synth.normal_bf16_bits(71, (nb, bs, hkv, d))
    lp = ops.LayerPointers([bf16_dev(cache_h, dev)])
    repre = torch.from_numpy(synth.normal_f32(72, (1, 20, hkv * d))).to(dev)
    before = repre.cpu().numpy().copy()
    ops.block_mean(lp, i32([9], dev), i32([13], dev), repre, bs, hkv, d, nb)
    after = repre.cpu().numpy()
    want = before.copy()
    O.block_mean_paged(cache_h, [9], [13], want[0])
    assert np.array_equal(bits(after), bits(want))
    assert not np.array_equal(bits(after[0, 13]), bits(before[0, 13]))


# ----------------------------------------------------------------- top-k

def run_topk(ops, dev, score_rows, topk, sw, ew, block_tables=None):
    lens = [len(s) for s in score_rows]
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    flat = np.concatenate([np.asarray(s, np.float32) for s in score_rows] + [np.zeros(1, np.float32)])
    scores = torch.from_numpy(flat[None]).to(dev)
    mx = max(max(lens), 1)
    idx = torch.full((1, len(lens), mx), -1, dtype=torch.int32, device=dev)
    cnt = torch.full((1, len(lens)), -1, dtype=torch.int32, device=dev)
    ops.topk_windows(scores, i32(off, dev), i32(lens, dev), i32(topk, dev), max(lens), idx, cnt, start_w=sw, end_w=ew)
    torch.cuda.synchronize()
    return idx.cpu().numpy()[0], cnt.cpu().numpy()[0]


def test_topk_golden_ties_on_gpu(ucm, dev, golden):
    from ucm_amd import ops

    z, meta = golden
    for i, n, k, sw, ew, seed in meta["ties"]:
        sc = synth.ints(seed, n, 0, 3).astype(np.float32)
        idx, cnt = run_topk(ops, dev, [sc], [k], sw, ew)
        want = z[f"ties/{i}"]
        assert cnt[0] == len(want) and np.array_equal(idx[0, : cnt[0]], want), (i, n, k, sw, ew)


@pytest.mark.parametrize("sw,ew", [(1, 2), (0, 0), (2, 0), (0, 3), (3, 5)])
def test_topk_many_requests_with_ties(ucm, dev, sw, ew):
    """Hundreds of small requests in one launch, scores drawn from four values so that
    almost every boundary is a tie; plus zeros of both signs and infinities."""
    from ucm_amd import ops

    rng = np.random.default_rng(80 + sw * 10 + ew)
    rows, ks = [], []
    for _ in range(300):
        n = int(rng.integers(1, 90))
        sc = rng.integers(-1, 3, n).astype(np.float32)
        sc[rng.random(n) < 0.1] = -0.0
        if rng.random() < 0.2:
            sc[rng.integers(0, n)] = np.inf
        if rng.random() < 0.2:
            sc[rng.integers(0, n)] = -np.inf
        rows.append(sc)
        ks.append(int(rng.integers(0, n + 3)))
    idx, cnt = run_topk(ops, dev, rows, ks, sw, ew)
    for r, sc in enumerate(rows):
        want = O.topk_windows(sc, ks[r], sw, ew)
        assert cnt[r] == len(want), (r, len(sc), ks[r])
        assert np.array_equal(idx[r, : cnt[r]], want), (r, len(sc), ks[r], sc)


@pytest.mark.parametrize("n", [64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4096])
def test_topk_register_tiers(ucm, dev, n):
    """Each register tier of the selection kernel (64, 128, ... 4096 blocks per request) at both of its ends."""
    from ucm_amd import ops

    sc = synth.normal_f32(90 + n, (n,))
    sc[::7] = sc[3]  # a large tie class that straddles the boundary for some k
    for k in (4, n // 3, n - 1):
        idx, cnt = run_topk(ops, dev, [sc, sc[: n // 2]], [k, k], 1, 2)
        for r, s in enumerate([sc, sc[: n // 2]]):
            want = O.topk_windows(s, k, 1, 2)
            assert cnt[r] == len(want) and np.array_equal(idx[r, : cnt[r]], want), (n, k, r)


# -------------------------------------------------------------- KV moves

def make_caches(dev, n_layers, nb, bb, seed):
    hs = [np.frombuffer(synth.u64(seed + l, 2 * nb * bb // 8).tobytes(), np.uint8).copy() for l in range(n_layers)]
    ds = [torch.from_numpy(h).to(dev) for h in hs]
    return hs, ds


def test_block_mean_of_large_launches_from_two_threads(ucm, dev):
    """Launches of one kernel that ask for LDS of different sizes, from two threads with streams of their own."""
    from ucm_amd import ops

    nb, bs, hkv, d = 16, 128, 8, 128
    cache = torch.empty((nb, bs, hkv, d), dtype=torch.bfloat16, device=dev).normal_()
    lp = ops.LayerPointers([cache])
    want = torch.zeros((1, nb, hkv * d), device=dev)
    ops.block_mean(lp, i32(np.arange(nb), dev), i32(np.arange(nb), dev), want, bs, hkv, d, nb)      # (another kernel: a small launch)
    torch.cuda.synchronize()
    faults = []

    def calls(n):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                ids = np.arange(n) % nb
                ids_d, slots = i32(ids, dev), i32(np.arange(n), dev)
                for _ in range(20):
                    out = torch.zeros((1, n, hkv * d), device=dev)
                    ops.block_mean(lp, ids_d, slots, out, bs, hkv, d, nb)
                    if not torch.equal(out[0], want[0, ids_d.long()]):
                        faults.append(n)
        except Exception as e:  # noqa: BLE001
            faults.append(repr(e))

    threads = [threading.Thread(target=calls, args=(n,)) for n in (1300, 12000)]                  # 3 and 24 groups a workgroup: 82 and 152 KiB
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not faults


@pytest.mark.parametrize("n", [5, 64, 128, 129, 256, 300, 512, 1000, 1024, 2048, 4096])
@pytest.mark.parametrize("kind", ["ties", "one value", "extremes", "all largest"])
def test_topk_windows_of_hard_scores(ucm, dev, n, kind):
    """Every tier of the selection where the threshold is shared: ties in index order, infinities, zeros of both signs, and
    NaNs up to the bit patterns whose keys are the smallest and the largest there are; none, one and most picks free."""
    from ucm_amd import ops

    rng = np.random.default_rng(n)
    pool = {"ties": np.array([0.5, -0.5, 1.5, 2.0], np.float32).view(np.uint32),
            "one value": np.array([0x3f800000], np.uint32),
            "extremes": np.array([0x7fffffff, 0xffffffff, 0x7f800000, 0xff800000, 0, 0x80000000, 0x3f800000], np.uint32),
            "all largest": np.array([0x7fffffff], np.uint32)}[kind]
    raw = rng.choice(pool, n).astype(np.uint32)
    u = np.where(raw == 0x80000000, 0, raw).astype(np.uint64)
    key = np.where(u >> 31, 0xffffffff - u, u | 0x80000000)
    sw, ew = 1, 2
    ks = [k for k in (sw + ew, sw + ew + 1, n // 3, n - 1) if sw + ew <= k < n]
    table = rng.permutation(n).astype(np.int32)
    scores = torch.from_numpy(np.tile(raw.view(np.int32), (len(ks), 1))).to(dev).view(torch.float32).contiguous()
    idx = torch.full((len(ks), 1, n), -7, dtype=torch.int32, device=dev)
    phys, cnt = idx.clone(), torch.zeros((len(ks), 1), dtype=torch.int32, device=dev)
    for l, k in enumerate(ks):
        one = slice(l, l + 1)
        ops.topk_windows(scores[one], i32([0], dev), i32([n], dev), i32([k], dev), n, idx[one], cnt[one], start_w=sw, end_w=ew,
                         block_tables=i32(table[None], dev), phys_out=phys[one])
    for l, k in enumerate(ks):
        middle = np.arange(sw, n - ew)
        best = middle[np.argsort(-key[middle].astype(np.int64), kind="stable")][: k - sw - ew]
        want = np.sort(np.concatenate([np.arange(sw), best, np.arange(n - ew, n)]))
        assert int(cnt[l, 0]) == k
        assert np.array_equal(idx[l, 0, :k].cpu().numpy(), want), (k, kind)
        assert np.array_equal(phys[l, 0, :k].cpu().numpy(), table[want])
        assert (idx[l, 0, k:] == -7).all()


@pytest.mark.parametrize("L,R,n", [(4, 256, 129), (5, 205, 129), (5, 205, 256), (4, 384, 257), (29, 53, 257), (29, 53, 512), (4, 384, 1000),
                                   (29, 53, 1000), (3, 513, 1024)])     # 1024 rows and more of up to 256 blocks, 1536 and more of longer ones
@pytest.mark.parametrize("kind", ["ties", "distinct", "extremes"])
def test_topk_windows_of_many_rows(ucm, dev, L, R, n, kind):
    """Both sides of the rule that gives a request one wave or four, every tier it covers, ragged lengths and numbers of picks."""
    from ucm_amd import ops

    rng = np.random.default_rng(n + R)
    if kind == "ties":
        scores = rng.integers(-6, 7, (L, R, n)).astype(np.float32)
    elif kind == "distinct":
        scores = rng.standard_normal((L, R, n)).astype(np.float32)
    else:
        scores = rng.choice(np.array([0x7fffffff, 0xffffffff, 0x7f800000, 0xff800000, 0, 0x3f800000], np.uint32), (L, R, n)).view(np.float32)
    lens = rng.integers(n // 2, n + 1, R).astype(np.int32)
    lens[0], lens[1] = n, 4
    ks = np.minimum(rng.integers(3, 40, R), lens - 1).astype(np.int32)
    table = np.argsort(rng.random((R, n)), axis=1).astype(np.int32)
    idx = torch.full((L, R, n), -7, dtype=torch.int32, device=dev)
    phys, cnt = idx.clone(), torch.zeros((L, R), dtype=torch.int32, device=dev)
    scores_d = torch.from_numpy(scores.view(np.int32)).to(dev).view(torch.float32).view(L, R * n)
    ops.topk_windows(scores_d, i32(np.arange(R) * n, dev), i32(lens, dev), i32(ks, dev), n, idx, cnt, block_tables=i32(table, dev), phys_out=phys)
    assert torch.equal(cnt, i32(ks, dev).expand(L, R))
    # the oracle's order by one sort over all rows: forced blocks first, then the candidates by key, the first index first
    u = scores.view(np.uint32).astype(np.int64)
    key = np.where(u >> 31, 0xffffffff - u, u | 0x80000000)
    i = np.arange(n)
    key[:, (i < 1) | ((i >= lens[:, None] - 2) & (i < lens[:, None]))] = 1 << 33
    key[:, i >= lens[:, None]] = -1
    order = np.argsort(-key, axis=-1, kind="stable")
    chosen = i < ks[:, None]
    want = np.sort(np.where(chosen, order, n), axis=-1)
    got, got_phys = idx.cpu().numpy(), phys.cpu().numpy()
    assert np.array_equal(np.where(want < n, want, -7), got)
    assert np.array_equal(np.where(want < n, table[np.arange(R)[None, :, None], np.minimum(want, n - 1)], -7), got_phys)


@pytest.mark.parametrize("L,R,longest", [(24, 32, 300), (25, 31, 300), (24, 64, 600), (29, 53, 600), (29, 53, 200)])   # 768, 775, 1536 and 1537 requests
@pytest.mark.parametrize("tile", [0, 2048])                              # tiles the library picks, and one for each request
def test_score_select_of_many_requests(ucm, dev, L, R, longest, tile):
    """Both sides of the rule that gives a request's selection one wave or four in the fused launch: what is selected is what the
    launch's own scores say, the first index of equal scores first."""
    from ucm_amd import ops

    rng = np.random.default_rng(R + longest)
    lens = rng.integers(4, longest + 1, R).astype(np.int32)
    lens[:6] = longest, 128, 129, min(longest, 256), min(longest, 257), 3
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    rows, ks = int(lens.sum()), np.minimum(rng.integers(4, 40, R), lens).astype(np.int32)
    q = torch.empty((L, R, 2, 64), dtype=torch.bfloat16, device=dev).normal_()
    repre = torch.empty((L, rows, 64), dtype=torch.bfloat16, device=dev).normal_()
    scores = torch.zeros((L, rows), device=dev)
    idx = torch.full((L, R, longest), -7, dtype=torch.int32, device=dev)
    cnt, tickets = torch.zeros((L, R), dtype=torch.int32, device=dev), torch.zeros((L, R), dtype=torch.int32, device=dev)
    for _ in range(2):                                                   # (the tickets are left as they were found)
        ops.score_select(q, repre, i32(off, dev), i32(lens, dev), i32(ks, dev), longest, 1, scores, idx, cnt, tickets, total_blocks=rows,
                         tile_blocks=tile)
    assert not tickets.any() and torch.equal(cnt, i32(ks, dev).expand(L, R))
    i = np.arange(longest)
    at = np.minimum(off[:, None] + i, rows - 1)
    s = scores.cpu().numpy()[:, at]
    s[:, (i < 1) | ((i >= lens[:, None] - 2) & (i < lens[:, None]))] = np.inf
    s[:, i >= lens[:, None]] = -np.inf
    order = np.argsort(-s, axis=-1, kind="stable")
    want = np.sort(np.where(i < ks[:, None], order, longest), axis=-1)
    assert np.array_equal(np.where(want < longest, want, -7), idx.cpu().numpy())


@pytest.mark.parametrize("bb", [262144, 4096, 48, 16 + 32768])
def test_kv_dump_load_round_trip(ucm, dev, bb):
    """Config-3 shape in small: random block table, scatter staging->cache, gather cache->staging, byte exact."""
    from ucm_amd import ops

    n_layers, nb, n = 3, 37, 11
    hs, ds = make_caches(dev, n_layers, nb, bb, 300)
    lp = ops.LayerPointers(ds)
    ids = synth.permutation(301, nb)[:n]
    staging = torch.zeros(n * n_layers * 2 * bb, dtype=torch.uint8, device=dev)
    ops.kv_gather_blocks(lp, nb * bb, bb, nb, i32(ids, dev), staging)
    want = np.zeros(n * n_layers * 2 * bb, np.uint8)
    O.kv_move_blocks(hs, nb * bb, bb, ids, want, True)
    assert np.array_equal(staging.cpu().numpy(), want)
    # load into a fresh cache: only the listed blocks change, and they equal the source
    fresh = [torch.zeros_like(t) for t in ds]
    lp2 = ops.LayerPointers(fresh)
    ops.kv_scatter_blocks(lp2, nb * bb, bb, nb, i32(ids, dev), staging)
    hfresh = [np.zeros_like(h) for h in hs]
    O.kv_move_blocks(hfresh, nb * bb, bb, ids, want, False)
    for l in range(n_layers):
        assert np.array_equal(fresh[l].cpu().numpy(), hfresh[l])
    # ids outside the plane are skipped
    ops.kv_gather_blocks(lp, nb * bb, bb, nb, i32([nb, -3], dev), staging)
    assert np.array_equal(staging.cpu().numpy(), want)


@pytest.mark.parametrize("bb", [16, 8192 - 16, 8192, 8192 + 16, 131072, 131072 + 16, 3 * 131072 + 8192 + 48])
def test_kv_moves_at_the_sizes_of_pieces(ucm, dev, bb):
    """Slices around what 256 threads take and around pieces of 128 KiB: dumps, loads and gathers of selected blocks, byte
    for byte, unusable ids and slots past the staging area left alone."""
    from ucm_amd import ops

    L, nb, n, n_req, stride = 2, 9, 5, 2, 4
    rng = np.random.default_rng(bb)
    host = rng.integers(0, 256, (L, 2, nb, bb), dtype=np.uint8)
    caches = [torch.from_numpy(host[l]).to(dev) for l in range(L)]
    lp, ids = ops.LayerPointers(caches), np.array([3, nb, 0, -1, 8], np.int32)
    staging = torch.full((n, L, 2, bb), 0xAB, dtype=torch.uint8, device=dev)
    ops.kv_gather_blocks(lp, nb * bb, bb, nb, i32(ids, dev), staging)
    want = np.full((n, L, 2, bb), 0xAB, np.uint8)
    for i in (0, 2, 4):
        want[i] = host[:, :, ids[i]]
    assert np.array_equal(staging.cpu().numpy(), want)
    to = np.array([1, nb, 7, -1, 2], np.int32)
    ops.kv_scatter_blocks(lp, nb * bb, bb, nb, i32(to, dev), staging)
    for i in (0, 2, 4):
        host[:, :, to[i]] = want[i]
    assert all(np.array_equal(caches[l].cpu().numpy(), host[l]) for l in range(L))
    phys = rng.integers(0, nb, (L, n_req, stride)).astype(np.int32)
    phys[0, 1, 1] = nb
    count = np.array([[3, 2], [4, 0]], np.int32)
    region = np.array([4, 2], np.int32)
    off = np.array([0, 4 * L * 2], np.int64)
    blocks = 6 * L * 2 - 1                                    # the last slot lies past the staging area
    out = torch.full((blocks + 1, bb), 0xCD, dtype=torch.uint8, device=dev)
    ops.kv_gather_selected(lp, nb * bb, bb, nb, i32(phys, dev), i32(count, dev), torch.from_numpy(off).to(dev), i32(region, dev),
                           stride, out, blocks)
    want = np.full((blocks + 1, bb), 0xCD, np.uint8)
    for l in range(L):
        for r in range(n_req):
            for kv in range(2):
                for j in range(count[l, r]):
                    slot = off[r] + (l * 2 + kv) * region[r] + j
                    if phys[l, r, j] < nb and slot < blocks:
                        want[slot] = host[l, kv, phys[l, r, j]]
    assert np.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("bb,n", [(131072, 3), (163840, 400), (196608, 64), (196608, 65),             # cut: 196608 x 64 only
                                  (262144, 64), (262144, 65), (262144, 128), (262144, 129), (262144, 384), (262144, 385),   # cut: 64, 129 and 385
                                  (262144 - 16, 385), (262144 + 16, 43), (262144 + 16, 100), (524288, 32), (524288, 100)])   # cut: all but the 100s
def test_kv_moves_of_cut_and_whole_slices(ucm, dev, bb, n):
    """Both sides of the rule that cuts a launch's slices between workgroups: dumps, loads, and gathers whose slots are all in use
    or nearly all idle (those stay whole), byte for byte."""
    from ucm_amd import ops

    nb = n + 3
    rng = np.random.default_rng(bb + n)
    gen = torch.Generator(device=dev)
    gen.manual_seed(n)
    cache = torch.randint(0, 256, (2, nb, bb), dtype=torch.uint8, device=dev, generator=gen)
    lp, ids = ops.LayerPointers([cache]), rng.permutation(nb)[:n].astype(np.int32)
    ids_d = i32(ids, dev)
    staging = torch.full((n, 1, 2, bb), 0xAB, dtype=torch.uint8, device=dev)
    ops.kv_gather_blocks(lp, nb * bb, bb, nb, ids_d, staging)
    want = cache[:, ids_d.long()].transpose(0, 1)
    assert torch.equal(staging[:, 0], want)
    to = rng.permutation(nb)[:n].astype(np.int32)
    loaded = cache.clone()
    ops.kv_scatter_blocks(ops.LayerPointers([loaded]), nb * bb, bb, nb, i32(to, dev), staging)
    after = cache.clone()
    after[:, i32(to, dev).long()] = want.transpose(0, 1)
    assert torch.equal(loaded, after)
    for used in (n, n // 9):                                                                # slots of the launch to blocks of the staging area
        out = torch.full((2 * used + 1, bb), 0xCD, dtype=torch.uint8, device=dev)
        ops.kv_gather_selected(lp, nb * bb, bb, nb, ids_d.view(1, 1, n), i32([[used]], dev), torch.zeros(1, dtype=torch.int64, device=dev),
                               i32([used], dev), n, out, 2 * used)
        assert torch.equal(out[: 2 * used].view(2, used, bb), cache[:, ids_d[:used].long()]) and (out[2 * used] == 0xCD).all()


def test_kv_moves_of_one_tensor_parallel_rank(ucm, dev):
    """Four ranks share the stored block; each moves its own K and V slices to where get_offset (esa.py:124-135) puts
    them, leaves the others' bytes alone, and reads them back - through the block moves and through the planned load."""
    from ucm_amd import ops

    n_layers, nb, n, tp, bb = 3, 23, 7, 4, 4096
    ids = synth.permutation(311, nb)[:n]
    staging = torch.full((n, n_layers * 2 * bb * tp), 0xEE, dtype=torch.uint8, device=dev)
    ranks = []
    for rank in range(tp):
        hs, ds = make_caches(dev, n_layers, nb, bb, 320 + rank)
        ranks.append((hs, ds))
        ops.kv_gather_blocks(ops.LayerPointers(ds), nb * bb, bb, nb, i32(ids, dev), staging, rank=rank, tp_size=tp)
        got = staging.cpu().numpy()
        for r2 in range(tp):                                         # ranks not yet written still hold the fill
            for l in range(n_layers):
                for kv in (0, 1):
                    at = O.get_offset((bb, 1, 1), r2, tp, 1, l, bool(kv))
                    for i, b in enumerate(ids):
                        piece = got[i, at : at + bb]
                        if r2 <= rank:
                            assert np.array_equal(piece, ranks[r2][0][l].reshape(2, nb, bb)[kv, b]), (rank, r2, l, kv, i)
                        else:
                            assert (piece == 0xEE).all()
    for rank in (2, 0):
        hs, _ = ranks[rank]
        fresh = [torch.zeros(2, nb, bb, dtype=torch.uint8, device=dev) for _ in range(n_layers)]
        ops.kv_scatter_blocks(ops.LayerPointers(fresh), nb * bb, bb, nb, i32(ids, dev), staging, rank=rank, tp_size=tp)
        # the planned load reads the same slices: logical block j of the one request is stored block j, slot j takes it
        planned = [torch.zeros(2, nb, bb, dtype=torch.uint8, device=dev) for _ in range(n_layers)]
        sel = torch.arange(n, dtype=torch.int32, device=dev).repeat(n_layers, 1, 1)
        src = torch.arange(n, dtype=torch.int32, device=dev).view(1, n)
        ops.kv_load_planned(ops.LayerPointers(planned), 0, 0, n_layers, nb * bb, bb, nb, staging, n_layers * 2 * bb * tp, sel, src,
                            i32(ids, dev).view(1, n), None, rank=rank, tp_size=tp)
        for l in range(n_layers):
            want = np.zeros((2, nb, bb), np.uint8)
            want[:, ids] = hs[l].reshape(2, nb, bb)[:, ids]
            assert np.array_equal(fresh[l].cpu().numpy(), want) and np.array_equal(planned[l].cpu().numpy(), want), (rank, l)
    with pytest.raises(ops.UcmHipError):
        ops.kv_gather_blocks(ops.LayerPointers(ranks[0][1]), nb * bb, bb, nb, i32(ids, dev), staging, rank=4, tp_size=4)


@pytest.mark.parametrize("n_slots,bb", [(1, 16), (64, 131072), (65, 131072 + 16), (1023, 48), (1024, 64), (1025, 16400), (40, 262144)])
def test_planned_loads_of_scattered_slots(ucm, dev, n_slots, bb):
    """Plans whose entries to load are scattered over a row: rows of up to, exactly and beyond the 1024 slots a workgroup lists
    at once, slices of less than a piece, one piece, a piece and sixteen bytes, two pieces; entries that are out of range
    anywhere, an empty row, a full row and a row outside the call's are left alone."""
    from ucm_amd import ops

    rng = np.random.default_rng(930 + n_slots)
    n_layers, rows_n, stored, src_n = 2, 4, 7, 9
    nb = n_slots + 3
    pool = rng.integers(0, 256, (stored, n_layers, 2, bb), dtype=np.uint8)
    load = np.where(rng.random((n_layers, rows_n, n_slots)) < 0.3, rng.integers(0, src_n, (n_layers, rows_n, n_slots)), -1).astype(np.int32)
    load[:, 1], load[0, 2] = -1, 5
    load[:, 0, 0] = src_n                                        # past the table of stored blocks
    src = rng.integers(0, stored, (rows_n, src_n)).astype(np.int32)
    src[:, 3], src[:, 4] = -1, stored                            # not in the pool
    dst = np.stack([rng.permutation(nb)[:n_slots] for _ in range(rows_n)]).astype(np.int32)
    dst[0, n_slots // 2] = nb
    for use in (np.array([2, -1, 0, 1, rows_n], np.int32), np.array([2], np.int32)):
        # one request's destinations at a time are distinct, those of several may meet: give each row a cache of its own
        for r in (use if len(use) == 1 else [2, 0]):
            caches = [torch.full((2, nb, bb), 0xEE, dtype=torch.uint8, device=dev) for _ in range(n_layers)]
            only = np.array([x if x in (r, -1, 1, rows_n) else -1 for x in use], np.int32)
            ops.kv_load_planned(ops.LayerPointers(caches), 0, 0, n_layers, nb * bb, bb, nb, torch.from_numpy(pool).to(dev).view(-1),
                                n_layers * 2 * bb, i32(load, dev), i32(src, dev), i32(dst, dev), i32(only, dev))
            for l in range(n_layers):
                want = np.full((2, nb, bb), 0xEE, np.uint8)
                for j in range(n_slots):
                    e = load[l, r, j]
                    if 0 <= e < src_n and 0 <= src[r, e] < stored and 0 <= dst[r, j] < nb:
                        want[:, dst[r, j]] = pool[src[r, e], l]
                assert np.array_equal(caches[l].cpu().numpy(), want), (r, l)


@pytest.mark.parametrize("counted", [False, True])
@pytest.mark.parametrize("n_layers,rows_n,n_slots,bb", [
    (2, 4, 9, 32768 + 16), (1, 3, 5, 32768), (1, 3, 7, 48), (2, 3, 5, 4 * 131072 + 4096),      # small launches, each size of workgroup
    (8, 9, 60, 65536), (8, 9, 60, 65536 + 16), (8, 9, 60, 131072), (8, 9, 60, 49152),          # large ones: a piece, a piece and a remainder, two
    (8, 9, 40, 131072 + 16), (4, 8, 40, 262144),                                              # the list: pieces of a longer slice
    (40, 41, 2, 48), (12, 40, 2, 131072 + 16),                                                # counts over several waves of the running total
    (65, 64, 3, 48), (65, 64, 1, 32768 + 16)])                                                # more rows than the counted kernel's table
def test_planned_loads_of_every_size_of_workgroup(ucm, dev, n_layers, rows_n, n_slots, bb, counted):
    """The rule that picks how a plan's loads are dealt out, on both sides of its bounds, with and without counts; with
    them a row's first entries load and what stands behind the count is left alone."""
    from ucm_amd import ops

    rng = np.random.default_rng(n_slots + bb)
    stored, src_n = 5, 6
    nb = rows_n * n_slots + 2
    pool = rng.integers(0, 256, (stored, n_layers, 2, bb), dtype=np.uint8)
    load = np.where(rng.random((n_layers, rows_n, n_slots)) < 0.4, rng.integers(0, src_n, (n_layers, rows_n, n_slots)), -1).astype(np.int32)
    count = rng.integers(-1, n_slots + 2, (n_layers, rows_n)).astype(np.int32)
    src = rng.integers(0, stored, (rows_n, src_n)).astype(np.int32)
    src[:, 2] = stored                                            # not in the pool
    dst = rng.permutation(nb)[: rows_n * n_slots].reshape(rows_n, n_slots).astype(np.int32)
    dst[rows_n // 2, 0] = nb
    caches = torch.full((n_layers, 2, nb, bb), 0xEE, dtype=torch.uint8, device=dev)
    ops.kv_load_planned(ops.LayerPointers([caches[l] for l in range(n_layers)]), 0, 0, n_layers, nb * bb, bb, nb,
                        torch.from_numpy(pool).to(dev).view(-1), n_layers * 2 * bb, i32(load, dev), i32(src, dev), i32(dst, dev), None,
                        load_count=i32(count, dev) if counted else None)
    pool_d = torch.from_numpy(pool).to(dev)
    for l in range(n_layers):
        want = torch.full((2, nb, bb), 0xEE, dtype=torch.uint8, device=dev)
        at, what = [], []
        for r in range(rows_n):
            for j in range(min(n_slots, max(int(count[l, r]), 0)) if counted else n_slots):
                e = load[l, r, j]
                if 0 <= e < src_n and src[r, e] < stored and dst[r, j] < nb:
                    at.append(int(dst[r, j]))
                    what.append(int(src[r, e]))
        if at:
            want[:, at] = pool_d[what, l].transpose(0, 1)
        assert torch.equal(caches[l], want), l


@pytest.mark.parametrize("n_layers,rows_n,n_slots,bb", [(32, 32, 2, 8192 + 16), (25, 41, 3, 16384), (40, 41, 2, 8192 + 16),   # a pair a thread, or four
                                                        (3, 5, 40, 3 * 131072 + 16), (2, 7, 6, 8192)])
def test_counted_loads_of_many_rows_and_long_slices(ucm, dev, n_layers, rows_n, n_slots, bb):
    """Running totals of 1024 pairs and more, slices of several pieces each, and a short plan of short slices, which goes by slot instead."""
    test_planned_loads_of_every_size_of_workgroup(ucm, dev, n_layers, rows_n, n_slots, bb, True)


@pytest.mark.parametrize("n_layers,rows_n,n_slots,bb", [
    (2, 16, 64, 4096), (2, 16, 65, 4096),                # 4096 slots to copy from, the last plan that goes slot by slot, and more
    (8, 20, 60, 16), (8, 20, 60, 1024 + 16), (8, 20, 60, 8192 - 16), (8, 20, 60, 8192),      # a wave's part of a slice, one trip of it and all
    (4, 64, 70, 64),                                     # more slices than there are waves
    (60, 68, 3, 48)])                                    # four pairs a thread in the running total
def test_counted_loads_of_short_slices(ucm, dev, n_layers, rows_n, n_slots, bb):
    """Slices of up to 8 KiB by single waves, on both sides of the rule that takes them."""
    test_planned_loads_of_every_size_of_workgroup(ucm, dev, n_layers, rows_n, n_slots, bb, True)


def test_copy_batch_pointer_arrays(ucm, dev):
    from ucm_amd import ops

    size, num = 65536 + 16, 9
    src = torch.from_numpy(np.frombuffer(synth.u64(310, num * size // 8).tobytes(), np.uint8).copy()).to(dev)
    dst = torch.zeros_like(src)
    order = synth.permutation(311, num).astype(np.int64)
    sp = torch.tensor([src.data_ptr() + int(i) * size for i in range(num)], dtype=torch.int64, device=dev)
    dp = torch.tensor([dst.data_ptr() + int(order[i]) * size for i in range(num)], dtype=torch.int64, device=dev)
    ops.copy_batch(dp, sp, size)
    got = dst.cpu().numpy().reshape(num, size)
    want = src.cpu().numpy().reshape(num, size)
    for i in range(num):
        assert np.array_equal(got[order[i]], want[i])
    ops.copy_batch(dp[:0], sp[:0], size)


def test_copy_batch_to_pinned_host(ucm, dev):
    """The staging side may be mapped pinned host memory (the reference's D2H kernel writes there)."""
    from ucm_amd import ops

    size, num = 8192, 5
    src = torch.from_numpy(np.frombuffer(synth.u64(320, num * size // 8).tobytes(), np.uint8).copy()).to(dev)
    host = torch.zeros(num * size, dtype=torch.uint8, pin_memory=True)
    sp = torch.tensor([src.data_ptr() + i * size for i in range(num)], dtype=torch.int64, device=dev)
    dp = torch.tensor([host.data_ptr() + i * size for i in range(num)], dtype=torch.int64, device=dev)
    ops.copy_batch(dp, sp, size)
    torch.cuda.synchronize()
    assert np.array_equal(host.numpy(), src.cpu().numpy())


def test_gather_selected_matches_oracle(ucm, dev):
    from ucm_amd import ops

    n_layers, nb, bb, n_req, stride = 4, 50, 8192, 3, 12
    hs, ds = make_caches(dev, n_layers, nb, bb, 330)
    lp = ops.LayerPointers(ds)
    count = synth.ints(331, n_layers * n_req, 0, 9).astype(np.int32).reshape(n_layers, n_req)
    phys = synth.ints(332, n_layers * n_req * stride, 0, nb - 1).astype(np.int32).reshape(n_layers, n_req, stride)
    region = count.max(0).astype(np.int32) + 1
    dst_off = np.concatenate([[0], np.cumsum(region * n_layers * 2)[:-1]]).astype(np.int64)
    total = int((region * n_layers * 2).sum())
    staging = torch.full((total * bb,), 0xAB, dtype=torch.uint8, device=dev)
    ops.kv_gather_selected(lp, nb * bb, bb, nb, i32(phys, dev), i32(count, dev),
                           torch.from_numpy(dst_off).to(dev), i32(region, dev), int(count.max()), staging, total)
    want = np.full(total * bb, 0xAB, np.uint8)
    O.kv_gather_selected(hs, nb * bb, bb, phys, count, dst_off, region, want)
    assert np.array_equal(staging.cpu().numpy(), want)

    # offsets that point past the staging buffer (they live in device memory, where the host cannot check them):
    # those destinations are skipped, everything else is written as before, nothing outside is touched
    guard = torch.full(((total + 4) * bb,), 0xCD, dtype=torch.uint8, device=dev)
    short = total - int(region[-1]) * 2                              # the last request's last layer does not fit
    bad_off = dst_off.copy()
    bad_off[0] = -5                                                   # and the first request points before the buffer
    ops.kv_gather_selected(lp, nb * bb, bb, nb, i32(phys, dev), i32(count, dev),
                           torch.from_numpy(bad_off).to(dev), i32(region, dev), int(count.max()), guard[: short * bb], short)
    got = guard.cpu().numpy()
    assert np.all(got[short * bb :] == 0xCD)
    first_len = int(region[0]) * n_layers * 2 * bb
    assert np.all(got[:first_len] == 0xCD)                            # request 0 was skipped entirely
    other = np.full(total * bb, 0x12, np.uint8)                       # a second background tells written bytes from the fill
    O.kv_gather_selected(hs, nb * bb, bb, phys, count, dst_off, region, other)
    written = (want == other)[first_len : short * bb]
    assert written.any() and np.array_equal(got[first_len : short * bb][written], want[first_len : short * bb][written])
    assert np.all(got[first_len : short * bb][~written] == 0xCD)


def test_retrieval_then_gather_end_to_end(ucm, dev):
    """Config-2 shape in small: means -> scores -> selection -> gather, no host round trip in between."""
    from ucm_amd import ops

    n_layers, hq, hkv, d, bs = 4, 32, 8, 128, 128
    lens = synth.ragged_lengths(340, 6, 4096, 16384)
    lens = np.minimum(lens, 60).astype(np.int32)
    topk = np.array([max(16, int(0.03 * n)) + 3 for n in lens], np.int32)
    nb = int(lens.sum()) + 4
    bb = bs * hkv * d * 2
    pairs = [randn_bf16(dev, 341 + l, (2, nb, bs, hkv, d)) for l in range(n_layers)]
    ds, caches_h = [p[0] for p in pairs], [p[1] for p in pairs]
    lp = ops.LayerPointers(ds)
    table = synth.permutation(350, nb)[: int(lens.sum())]
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    rows = int(lens.sum())
    repre = torch.zeros(n_layers, rows, hkv * d, device=dev)
    ops.block_mean(lp, i32(table, dev), i32(np.arange(rows), dev), repre, bs, hkv, d, nb)
    q = synth.normal_bf16_as_f32(351, (n_layers, len(lens), hq, d))
    bt = np.zeros((len(lens), int(lens.max())), np.int32)
    for r, n in enumerate(lens):
        bt[r, :n] = table[off[r] : off[r] + n]
    repre_h = repre.cpu().numpy()
    out = run_select(ops, dev, q, repre_h, lens, topk, hkv, q_dtype=torch.bfloat16, block_tables=bt)
    check_against_oracle(out, q, repre_h, lens, topk, hkv)
    for l in range(n_layers):
        want_rep = np.zeros((rows, hkv * d), np.float32)
        O.block_mean_paged(caches_h[l][0], table, np.arange(rows), want_rep)
        assert np.array_equal(bits(repre_h[l]), bits(want_rep))
    region = topk.copy()
    dst_off = np.concatenate([[0], np.cumsum(region.astype(np.int64) * n_layers * 2)[:-1]]).astype(np.int64)
    total = int((region.astype(np.int64) * n_layers * 2).sum())
    staging = torch.zeros(total * bb, dtype=torch.uint8, device=dev)
    ops.kv_gather_selected(lp, nb * bb, bb, nb, i32(out["phys"], dev), i32(out["cnt"], dev),
                           torch.from_numpy(dst_off).to(dev), i32(region, dev), int(topk.max()), staging, total)
    want = np.zeros(total * bb, np.uint8)
    O.kv_gather_selected([c.view(np.uint8).reshape(-1) for c in caches_h], nb * bb, bb, out["phys"], out["cnt"],
                         dst_off, region, want)
    assert np.array_equal(staging.cpu().numpy(), want)


# ------------------------------------------- the benchmark configurations at full size

def test_config3_full_size_round_trip(ucm, dev):
    """64 requests x 2048-token budget (16 blocks) x 32 layers, K and V: 17.2 GB per direction.  A random block
    table over the pool drives the load (staging -> cache) and the dump (cache -> staging); the round trip must be
    byte exact and the rest of the pool untouched.  (The literal 200k-block pool x 32 layers would be 3.4 TB; the
    pool here is 4096 blocks per layer, 68.7 GB, which does not change what the kernels do.)"""
    from ucm_amd import ops

    free, _ = torch.cuda.mem_get_info()
    if free < 120 * 2 ** 30:
        pytest.skip("needs about 105 GB of free HBM")
    n_layers, nb, bb, n = 32, 4096, 262144, 64 * 16
    caches = [torch.zeros(2 * nb * bb, dtype=torch.uint8, device=dev) for _ in range(n_layers)]
    lp = ops.LayerPointers(caches)
    ids_h = synth.permutation(400, nb)[:n]
    ids = i32(ids_h, dev)
    g = torch.Generator(device=dev)
    g.manual_seed(401)
    src = torch.empty(n * n_layers * 2 * bb // 8, dtype=torch.int64, device=dev)
    src.random_(generator=g)
    src = src.view(torch.uint8)
    ops.kv_scatter_blocks(lp, nb * bb, bb, nb, ids, src)
    back = torch.zeros_like(src)
    ops.kv_gather_blocks(lp, nb * bb, bb, nb, ids, back)
    torch.cuda.synchronize()
    assert torch.equal(src, back)
    # spot checks of placement against the closed form, and nothing outside the listed blocks was written
    sv = src.view(n, n_layers, 2, bb)
    for (i, l, kv) in [(0, 0, 0), (5, 31, 1), (n - 1, 17, 0)]:
        assert torch.equal(caches[l].view(2, nb, bb)[kv, int(ids_h[i])], sv[i, l, kv])
    untouched = torch.ones(nb, dtype=torch.bool, device=dev)
    untouched[ids.long()] = False
    for l in (0, 13, 31):
        assert not caches[l].view(2, nb, bb)[:, untouched].any()


def test_config4_full_size_selection(ucm, dev):
    """Qwen2-72B shape at full size: 8 requests of 512-1024 blocks, 80 layers, 64 query heads (g = 8),
    k = 2 % + windows: every score and every selected index against the oracle."""
    from ucm_amd import ops

    n_layers, hkv, g, d = 80, 8, 8, 128
    lens = synth.ragged_lengths(410, 8, 65536, 131072)
    topk = np.array([max(16, int(0.02 * n)) + 3 for n in lens], np.int32)
    rows = int(lens.sum())
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    gen = torch.Generator(device=dev)
    gen.manual_seed(411)
    repre = torch.randn(n_layers, rows, hkv * d, device=dev, generator=gen)
    q = torch.randn(n_layers, len(lens), hkv * g, d, device=dev, generator=gen).to(torch.bfloat16)
    scores = torch.zeros(n_layers, rows, device=dev)
    ops.score_blocks(q, repre, i32(off, dev), i32(lens, dev), int(lens.max()), hkv, scores, total_blocks=rows)
    idx = torch.full((n_layers, len(lens), int(lens.max())), -1, dtype=torch.int32, device=dev)
    cnt = torch.zeros(n_layers, len(lens), dtype=torch.int32, device=dev)
    ops.topk_windows(scores, i32(off, dev), i32(lens, dev), i32(topk, dev), int(lens.max()), idx, cnt)
    torch.cuda.synchronize()
    q_h, rep_h = q.float().cpu().numpy(), repre.cpu().numpy()
    sc_h, idx_h, cnt_h = scores.cpu().numpy(), idx.cpu().numpy(), cnt.cpu().numpy()
    for l in range(n_layers):
        widx, wcnt, wsc = O.select_topk_bs(q_h[l], rep_h[l], off, lens, topk, hkv, out_stride=int(lens.max()) + 4)
        assert np.array_equal(bits(sc_h[l]), bits(wsc)), l
        assert np.array_equal(cnt_h[l], wcnt), l
        for r in range(len(lens)):
            assert np.array_equal(idx_h[l, r, : wcnt[r]], widx[r, : wcnt[r]]), (l, r)


def test_delta_plan_and_delta_gather(ucm, dev):
    """Several decode steps of changing selections: the plan matches the oracle, only missing blocks move,
    and after every step each request's staging slots hold exactly the selected blocks."""
    from ucm_amd import ops

    n_layers, n_req, n_slots, nb, bb, stride = 3, 5, 19, 300, 4096, 40
    hs, ds = make_caches(dev, n_layers, nb, bb, 500)
    lp = ops.LayerPointers(ds)
    resident = torch.full((n_layers, n_req, n_slots), -1, dtype=torch.int32, device=dev)
    res_h = np.full((n_layers, n_req, n_slots), -1, np.int32)
    region = np.full(n_req, n_slots, np.int32)
    dst_off = (np.arange(n_req, dtype=np.int64) * n_slots * n_layers * 2)
    total = n_req * n_slots * n_layers * 2
    staging = torch.zeros(total * bb, dtype=torch.uint8, device=dev)
    tables = np.stack([synth.permutation(510 + r, nb)[:50] for r in range(n_req)]).astype(np.int32)   # logical -> cache block
    slots_count = i32(np.full((n_layers, n_req), n_slots), dev)
    rng = np.random.default_rng(12)
    prev = None
    for step in range(6):
        cnt = rng.integers(0, n_slots + 1, (n_layers, n_req)).astype(np.int32)
        cnt[0, 0] = n_slots
        sel = np.full((n_layers, n_req, stride), -1, np.int32)
        for l in range(n_layers):
            for r in range(n_req):
                if prev is not None and rng.random() < 0.7:       # mostly overlapping with the previous step
                    base = set(prev[l, r][prev[l, r] >= 0].tolist())
                    pool = list(base) + list(rng.permutation(50)[:6])
                    pick = np.unique(np.array(pool))[: cnt[l, r]]
                    rng.shuffle(pick)
                    pick = np.sort(pick[: cnt[l, r]])
                else:
                    pick = np.sort(rng.permutation(50)[: cnt[l, r]])
                cnt[l, r] = len(pick)
                sel[l, r, : len(pick)] = pick
        phys = np.where(sel >= 0, np.take_along_axis(np.broadcast_to(tables[None], (n_layers, n_req, 50)),
                                                      np.maximum(sel, 0), axis=2), -1).astype(np.int32)
        load = torch.full((n_layers, n_req, n_slots), -7, dtype=torch.int32, device=dev)
        slot_of = torch.full((n_layers, n_req, stride), -7, dtype=torch.int32, device=dev)
        miss = torch.full((n_layers, n_req), -7, dtype=torch.int32, device=dev)
        ops.delta_plan(i32(sel, dev), i32(phys, dev), i32(cnt, dev), resident, load, slot_of, miss)
        ops.kv_gather_selected(lp, nb * bb, bb, nb, load, slots_count, torch.from_numpy(dst_off).to(dev),
                               i32(region, dev), n_slots, staging, total)
        torch.cuda.synchronize()
        load_h, slot_h, miss_h, st = load.cpu().numpy(), slot_of.cpu().numpy(), miss.cpu().numpy(), staging.cpu().numpy()
        for l in range(n_layers):
            for r in range(n_req):
                k = int(cnt[l, r])
                wl, ws, moved = O.delta_plan(sel[l, r, :k], phys[l, r, :k], res_h[l, r])
                assert np.array_equal(load_h[l, r], wl) and miss_h[l, r] == moved, (step, l, r)
                assert np.array_equal(slot_h[l, r, :k], ws), (step, l, r)
                # every selected block is now in its slot, K and V
                for i in range(k):
                    for kv in range(2):
                        o = (int(dst_off[r]) + (l * 2 + kv) * n_slots + int(ws[i])) * bb
                        src = hs[l].reshape(2, nb, bb)[kv, phys[l, r, i]]
                        assert np.array_equal(st[o : o + bb], src), (step, l, r, i, kv)
        assert np.array_equal(resident.cpu().numpy(), res_h)
        if step > 0:
            assert miss_h.sum() < cnt.sum()        # overlapping selections really save loads
        prev = sel


@pytest.mark.parametrize("n_slots", [1, 63, 64, 65, 153, 256, 257, 512, 700, 1024])
def test_delta_plan_slot_counts(ucm, dev, n_slots):
    """The plan for one to 1024 staging slots (one wave up to 64, a workgroup beyond) over four steps of
    drifting selections in score order (not ascending), with counts from empty to beyond the slot budget,
    equals the oracle's: loads, slot of every selected block, resident sets, counts."""
    from ucm_amd import ops

    n_layers, n_req = 2, 3
    universe = 2 * n_slots + 40
    stride = n_slots + 9
    rng = np.random.default_rng(1000 + n_slots)
    resident = torch.full((n_layers, n_req, n_slots), -1, dtype=torch.int32, device=dev)
    res_h = np.full((n_layers, n_req, n_slots), -1, np.int32)
    table = rng.permutation(5 * universe)[:universe].astype(np.int32)
    prev = [[None] * n_req for _ in range(n_layers)]
    for step in range(4):
        cnt = rng.integers(0, stride + 1, (n_layers, n_req)).astype(np.int32)
        cnt[0, 0], cnt[1, 1] = min(stride, n_slots + 5), n_slots
        if step == 2:
            cnt[0, 2] = 0
        sel = np.full((n_layers, n_req, stride), -1, np.int32)
        for l in range(n_layers):
            for r in range(n_req):
                c = int(cnt[l, r])
                if prev[l][r] is not None and len(prev[l][r]):
                    old = prev[l][r]
                    keep = old[rng.random(len(old)) < 0.8]
                    fresh = np.setdiff1d(rng.permutation(universe), keep, assume_unique=True)
                    pick = np.concatenate([keep, fresh])[:c]
                else:
                    pick = rng.permutation(universe)[:c]
                pick = rng.permutation(pick).astype(np.int32)
                sel[l, r, :c] = pick
                prev[l][r] = pick
        phys = np.where(sel >= 0, table[np.maximum(sel, 0)], -1).astype(np.int32)
        load = torch.full((n_layers, n_req, n_slots), -7, dtype=torch.int32, device=dev)
        slot_of = torch.full((n_layers, n_req, stride), -7, dtype=torch.int32, device=dev)
        miss = torch.full((n_layers, n_req), -7, dtype=torch.int32, device=dev)
        ops.delta_plan(i32(sel, dev), i32(phys, dev), i32(cnt, dev), resident, load, slot_of, miss)
        torch.cuda.synchronize()
        load_h, slot_h, miss_h = load.cpu().numpy(), slot_of.cpu().numpy(), miss.cpu().numpy()
        for l in range(n_layers):
            for r in range(n_req):
                c = int(cnt[l, r])
                wl, ws, moved = O.delta_plan(sel[l, r, :c], phys[l, r, :c], res_h[l, r])
                k = min(c, n_slots)
                assert np.array_equal(load_h[l, r], wl) and miss_h[l, r] == moved, (step, l, r)
                assert np.array_equal(slot_h[l, r, :k], ws[:k]), (step, l, r)
                assert np.all(slot_h[l, r, k:] == -7), (step, l, r)      # nothing written past the cut
        assert np.array_equal(resident.cpu().numpy(), res_h), step


@pytest.mark.parametrize("n_layers,n_req", [(64, 8), (57, 9)])
@pytest.mark.parametrize("n_slots", [65, 256, 257, 530])
def test_delta_plan_on_both_sides_of_the_thread_split(ucm, dev, n_layers, n_req, n_slots):
    """512 rows (four threads per entry of 256 slots, one otherwise) and 513 (one), with slots that hold a block twice or nothing: the last slot of a
    block wins, and loads, slots, resident sets and counts equal the oracle's."""
    from ucm_amd import ops

    rng = np.random.default_rng(n_slots + n_req)
    sel = np.stack([rng.permutation(2 * n_slots)[: n_slots + 3] for _ in range(n_layers * n_req)]).astype(np.int32)
    sel = sel.reshape(n_layers, n_req, -1)
    cnt = rng.integers(0, n_slots + 4, (n_layers, n_req)).astype(np.int32)
    cnt[0, 0], cnt[-1, -1] = 0, n_slots
    res_h = rng.integers(-1, 2 * n_slots, (n_layers, n_req, n_slots)).astype(np.int32)
    resident, phys = i32(res_h, dev), sel + 7
    load = torch.full((n_layers, n_req, n_slots), -7, dtype=torch.int32, device=dev)
    slot_of, miss = i32(np.full_like(sel, -7), dev), i32(np.full_like(cnt, -7), dev)
    ops.delta_plan(i32(sel, dev), i32(phys, dev), i32(cnt, dev), resident, load, slot_of, miss)
    load_h, slot_h, miss_h = load.cpu().numpy(), slot_of.cpu().numpy(), miss.cpu().numpy()
    for l in range(n_layers):
        for r in range(n_req):
            c = int(cnt[l, r])
            wl, ws, moved = O.delta_plan(sel[l, r, :c], phys[l, r, :c], res_h[l, r])
            k = min(c, n_slots)
            assert np.array_equal(load_h[l, r], wl) and miss_h[l, r] == moved, (l, r)
            assert np.array_equal(slot_h[l, r, :k], ws[:k]) and np.all(slot_h[l, r, k:] == -7), (l, r)
    assert np.array_equal(resident.cpu().numpy(), res_h)


@pytest.mark.parametrize("n_layers,n_req,n_slots", [(32, 8, 65), (1, 257, 99), (1, 257, 100), (57, 9, 100), (32, 8, 257), (1, 257, 299), (64, 8, 300),
                                                    (32, 8, 513), (1, 257, 831), (64, 8, 832), (57, 9, 832)])
def test_delta_plan_of_longer_walks_on_both_sides_of_the_thread_split(ucm, dev, n_layers, n_req, n_slots):
    """256 rows always have four threads per entry, up to 512 only with enough slots."""
    test_delta_plan_on_both_sides_of_the_thread_split(ucm, dev, n_layers, n_req, n_slots)


def test_decode_step_under_graph_capture(ucm, dev):
    """The step's three launches (scores, selection + block table, gather) allocate and synchronise nothing, so a
    caller may capture them in a HIP graph: three replays with fresh queries, eager work and synchronisation in
    between, each equal to the eager result for the same queries."""
    from ucm_amd import ops

    n_layers, hq, hkv, d, bs = 3, 32, 8, 128, 16
    lens = np.array([40, 7, 25, 3], np.int32)
    topk = np.array([19, 7, 19, 3], np.int32)
    rows, nb = int(lens.sum()), int(lens.sum()) + 3
    bb = bs * hkv * d * 2
    caches = [randn_bf16(dev, 1700 + l, (2, nb, bs, hkv, d))[0] for l in range(n_layers)]
    lp = ops.LayerPointers(caches)
    table = synth.permutation(1710, nb)[:rows]
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    repre = torch.zeros(n_layers, rows, hkv * d, device=dev, dtype=torch.bfloat16)
    ops.block_mean(lp, i32(table, dev), i32(np.arange(rows), dev), repre, bs, hkv, d, nb, mode=ops.MEAN_BF16_STORE)
    bt = np.zeros((len(lens), int(lens.max())), np.int32)
    for r, n in enumerate(lens):
        bt[r, :n] = table[off[r] : off[r] + n]
    mx, kmax = int(lens.max()), int(topk.max())
    seg_off, seg_len, topk_d, bt_d = i32(off, dev), i32(lens, dev), i32(topk, dev), i32(bt, dev)
    region = i32(topk, dev)
    dst_off = torch.from_numpy(np.concatenate([[0], np.cumsum(topk.astype(np.int64) * n_layers * 2)[:-1]])).to(dev)
    total = int((topk.astype(np.int64) * n_layers * 2).sum())

    def buffers():
        return (torch.full((n_layers, rows), -5.0, device=dev), torch.full((n_layers, len(lens), mx), -1, dtype=torch.int32, device=dev),
                torch.full((n_layers, len(lens)), -1, dtype=torch.int32, device=dev),
                torch.full((n_layers, len(lens), mx), -1, dtype=torch.int32, device=dev),
                torch.full((total * bb,), 7, dtype=torch.uint8, device=dev))

    def step(q, scores, idx, cnt, phys, staging):
        ops.score_blocks(q, repre, seg_off, seg_len, mx, hkv, scores)
        ops.topk_windows(scores, seg_off, seg_len, topk_d, mx, idx, cnt, block_tables=bt_d, phys_out=phys)
        ops.kv_gather_selected(lp, nb * bb, bb, nb, phys, cnt, dst_off, region, kmax, staging, total)

    q_static = torch.zeros(n_layers, len(lens), hq, d, device=dev, dtype=torch.bfloat16)
    g_bufs = buffers()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(q_static, *g_bufs)                                   # warm-up outside the capture
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(q_static, *g_bufs)
    for rep in range(3):
        q = torch.from_numpy(synth.normal_bf16_as_f32(1720 + rep, (n_layers, len(lens), hq, d))).to(dev).to(torch.bfloat16)
        e_bufs = buffers()
        step(q, *e_bufs)                                          # eager, on the current stream
        torch.cuda.synchronize()
        q_static.copy_(q)
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip(("scores", "idx", "cnt", "phys", "staging"), g_bufs, e_bufs):
            assert torch.equal(a, b), (rep, name)
        assert int(e_bufs[2].min()) > 0                           # something was selected for every request


def test_device_and_host_twins_give_the_same_bytes(ucm, dev):
    """One scripted pass over the dense path (three representative modes, both score variants with q_rows and a
    scale, selection with block tables and sparse lengths, two delta plans, both gathers, block moves with ids to
    skip; the hash-code path; the ESA worker's retrieval, batched and over a persistent table, with two plans of its
    winners) through libucm_hip.so on device buffers and through the oracle's `_cpu` twins on host buffers: the same
    argument lists, the same bytes out."""
    import cpu_twins
    from ucm_amd import _lib, ops

    # the dense path; descriptors outside the tables; hash codes; the ESA worker; KVStar's selection, prefetch round, planned loads
    for run in (cpu_twins.run, cpu_twins.run_bounds, cpu_twins.run_hash, cpu_twins.run_esa, cpu_twins.run_more):
        want, _ = run(cpu_twins.twin_caller(_lib.SIGNATURES), cpu_twins.HostSide())
        got, _ = run(_lib.call, cpu_twins.DeviceSide(ops, dev))
        assert got.keys() == want.keys()
        for name in want:
            assert got[name].dtype == want[name].dtype and got[name].shape == want[name].shape, name
            assert np.array_equal(got[name].view(np.uint8), want[name].view(np.uint8)), name
    # KVStar: the tables bit for bit; the votes to rounding (the matrix cores sum in another order than the scalar loop)
    want, _ = cpu_twins.run_kvstar(cpu_twins.twin_caller(_lib.SIGNATURES), cpu_twins.HostSide())
    got, _ = cpu_twins.run_kvstar(_lib.call, cpu_twins.DeviceSide(ops, dev))
    for name in ("table_full", "table_pruned", "table_by_block", "park_f32", "park_bf16", "park_f16", "rows_indexed", "rows_in_order"):
        assert np.array_equal(got[name], want[name]), name
    for name in ("votes", "votes_tables", "votes_bad0", "votes_bad1", "votes_bad2"):
        assert np.allclose(got[name], want[name], rtol=2e-4, atol=2e-6), name
        assert np.array_equal(got[name] == -3, want[name] == -3), name        # the same tasks were skipped


def test_device_and_host_twins_on_other_seeds(ucm, dev):
    """The scripted passes of the test above on inputs drawn from other seeds - 150 sets by default,
    UCM_TWIN_SEED_SETS of them when that is set (6000 sets take three minutes) - with the same comparison."""
    import os

    import cpu_twins
    from ucm_amd import _lib, ops

    exact = ("table_full", "table_pruned", "table_by_block", "park_f32", "park_bf16", "park_f16", "rows_indexed", "rows_in_order")
    for it in range(1, int(os.environ.get("UCM_TWIN_SEED_SETS", "150")) + 1):
        with cpu_twins.reseeded(it * 100003):
            for run in (cpu_twins.run, cpu_twins.run_bounds, cpu_twins.run_hash, cpu_twins.run_esa, cpu_twins.run_more):
                want, _ = run(cpu_twins.twin_caller(_lib.SIGNATURES), cpu_twins.HostSide())
                got, _ = run(_lib.call, cpu_twins.DeviceSide(ops, dev))
                for name in want:
                    assert np.array_equal(got[name].view(np.uint8), want[name].view(np.uint8)), (it, run.__name__, name)
            want, _ = cpu_twins.run_kvstar(cpu_twins.twin_caller(_lib.SIGNATURES), cpu_twins.HostSide())
            got, _ = cpu_twins.run_kvstar(_lib.call, cpu_twins.DeviceSide(ops, dev))
        for name in exact:
            assert np.array_equal(got[name], want[name]), (it, name)
        for name in ("votes", "votes_tables", "votes_bad0", "votes_bad1", "votes_bad2"):
            assert np.allclose(got[name], want[name], rtol=2e-4, atol=2e-6), (it, name)


@pytest.mark.parametrize("dtype,row", [("bfloat16", (32, 128)), ("float32", (8, 64)), ("float16", (3, 8))])
def test_park_rows_against_torch_indexing(ucm, dev, dtype, row):
    """ucm_park_rows: rows of a query tensor into rows of a kept-queries table, picked and placed by device index
    arrays - a thousand pairs, some naming rows outside either array (skipped), with and without destination
    indices - against torch's own indexing."""
    from ucm_amd import ops

    dt = getattr(torch, dtype)
    g = torch.Generator(device=dev)
    g.manual_seed(77)
    src = torch.randn((700,) + row, device=dev, generator=g).to(dt)
    dst = torch.full((1000,) + row, 3.0, dtype=dt, device=dev)
    rng = np.random.default_rng(78)
    pick = rng.integers(-5, 710, 1000).astype(np.int32)                  # a few below 0, a few past the end
    put = rng.permutation(1010)[:1000].astype(np.int32) - 3              # distinct; a few outside [0, 1000)
    ops.park_rows(src, torch.from_numpy(pick).to(dev), dst, torch.from_numpy(put).to(dev))
    want = torch.full_like(dst, 3.0)
    ok = (pick >= 0) & (pick < 700) & (put >= 0) & (put < 1000)
    want[torch.from_numpy(put[ok].astype(np.int64)).to(dev)] = src[torch.from_numpy(pick[ok].astype(np.int64)).to(dev)]
    assert 900 < ok.sum() < 1000 and torch.equal(dst.view(torch.uint8), want.view(torch.uint8))
    dst2 = torch.full((1000,) + row, 3.0, dtype=dt, device=dev)
    ops.park_rows(src, torch.from_numpy(pick).to(dev), dst2)            # pair i goes to row i
    want2 = torch.full_like(dst2, 3.0)
    ok2 = (pick >= 0) & (pick < 700)
    at = torch.from_numpy(np.nonzero(ok2)[0]).to(dev)
    want2[at] = src[torch.from_numpy(pick[ok2].astype(np.int64)).to(dev)]
    assert torch.equal(dst2.view(torch.uint8), want2.view(torch.uint8))
    with pytest.raises(ValueError):
        ops.park_rows(src, torch.from_numpy(pick).to(dev), dst.float() if dt != torch.float32 else dst.half())
