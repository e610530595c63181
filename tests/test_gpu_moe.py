"""GPU parity of the fused-MoE pieces against the CPU oracle (exact for routing / align,
2e-3 relative Frobenius for the block output)."""
import os

import numpy as np
import pytest
import torch

from oracle import awq_ref

pytestmark = pytest.mark.gpu
TOL = 2e-3
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


@pytest.mark.parametrize("T,E,topk", [(1, 128, 8), (16, 128, 8), (128, 128, 8), (512, 128, 8), (7, 4, 2),
                                      (33, 1024, 6), (5, 64, 64)])
def test_topk_softmax(sba, gpu, T, E, topk):
    g = torch.Generator().manual_seed(T + E)
    logits = torch.randn((T, E), generator=g)
    for renorm in (True, False):
        w, ids = sba.topk_softmax(logits.to(gpu), topk, renorm)
        rid, rw = awq_ref.topk_softmax(logits.numpy(), topk, renorm)
        assert np.array_equal(ids.cpu().numpy(), rid)
        assert np.allclose(w.cpu().numpy(), rw, rtol=2e-5, atol=1e-8)
    tie = torch.zeros((2, E))
    _, ids = sba.topk_softmax(tie.to(gpu), topk, True)
    assert ids.cpu().tolist() == [list(range(topk))] * 2


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("T,E,topk", [(1, 16, 16), (3, 17, 16), (5, 60, 1), (4, 64, 8), (9, 65, 8), (17, 127, 6), (6, 128, 16),
                                      (7, 129, 4), (2, 255, 16), (18, 256, 8), (5, 257, 16), (5, 128, 17), (1, 1, 1)])
def test_topk_with_many_ties_at_the_edges_of_its_forms(sba, gpu, scoring, T, E, topk):
    """Experts and picks on both sides of what sixteen lanes a token hold (256 and 16), tokens that leave part of a wave
    empty, rows that are no multiple of 16 bytes; logits of few values, zeros of both signs among them, so that ties lie inside
    a lane, across lanes and across the experts' whole range."""
    g = torch.Generator().manual_seed(31 * T + E + topk)
    logits = torch.randint(-2, 3, (T, E), generator=g).float()
    logits[torch.rand((T, E), generator=g) < 0.3] *= -0.0
    if scoring == "softmax":
        w, ids = sba.topk_softmax(logits.to(gpu), topk, True)
        rid, rw = awq_ref.topk_softmax(logits.numpy(), topk, True)
    else:
        # (of a few values too: the scores of equal logits are equal)
        bias = torch.randint(0, 2, (E,), generator=g).float()
        w, ids = sba.topk_route(logits.to(gpu), topk, True, "sigmoid", bias.to(gpu))
        rid, rw = awq_ref.topk_sigmoid(logits.numpy(), topk, True, bias.numpy())
    assert np.array_equal(ids.cpu().numpy(), rid)
    assert np.allclose(w.cpu().numpy(), rw, rtol=2e-5, atol=1e-8)


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
def test_topk_with_nan_and_infinite_logits_keeps_ids_in_range(sba, gpu, scoring):
    """Rows with fewer than top-k usable logits: NaN keys lose against every number and are then
    taken in expert order (the oracle's stable argsort puts them last the same way), -inf keys
    tie towards the lowest id.  Every id must be a distinct expert inside [0, E) - an id of E
    would leave that slot's rows unwritten - and the block built on such routing must still
    write every output row.  (How vLLM's own routing kernel orders NaN keys is not pinned by
    anything available here; the weights of such rows are NaN on both sides.)"""
    E, topk = 128, 8
    lg = torch.randn((6, E), generator=torch.Generator().manual_seed(1))
    lg[0, 5:] = float("nan")                 # five numbers, the rest NaN
    lg[1, :] = float("nan")                  # nothing usable
    lg[2, :] = float("-inf")                 # all tied at -inf
    lg[3, 3:] = float("-inf")                # three numbers, the rest -inf
    lg[4, ::2] = float("nan")                # every other one NaN
    if scoring == "softmax":
        w, ids = sba.topk_softmax(lg.to(gpu), topk, True)
        rid, rw = awq_ref.topk_softmax(lg.numpy(), topk, True)
    else:
        w, ids = sba.topk_route(lg.to(gpu), topk, True, "sigmoid")
        rid, rw = awq_ref.topk_sigmoid(lg.numpy(), topk, True)
    ids, w = ids.cpu().numpy(), w.cpu().numpy()
    assert ids.min() >= 0 and ids.max() < E
    assert all(len(set(r.tolist())) == topk for r in ids)
    assert np.array_equal(ids, rid)
    assert np.allclose(w, rw, rtol=2e-5, atol=1e-8, equal_nan=True)
    assert np.isfinite(w[5]).all() and np.isfinite(w[3]).all() and np.isnan(w[[0, 1]]).all()
    if scoring == "softmax":
        assert np.isnan(w[[2, 4]]).all()
        c = sba.workloads.make_moe_case(6, 256, E, topk, 128, 128, seed=4).to(gpu)
        y = sba.fused_moe_awq(c.x, c.w13, c.w2, lg.to(gpu), topk, True)
        torch.cuda.synchronize()
        assert torch.isfinite(y[5]).all() and torch.isfinite(y[3]).all()      # rows with usable routing
        assert torch.isnan(y[[0, 1, 2, 4]]).all()      # NaN weights reach every element: no row is stale


@pytest.mark.parametrize("T,E,topk,tile", [(1, 128, 8, 16), (16, 128, 8, 16), (512, 128, 8, 16), (7, 4, 2, 4),
                                           (1000, 8, 2, 16), (64, 1024, 4, 16), (3, 5, 1, 1), (4096, 128, 8, 16)])
def test_moe_align_equals_oracle(sba, gpu, T, E, topk, tile):
    rng = np.random.default_rng(T * 7 + E)
    ids = np.stack([rng.choice(E, size=topk, replace=False) for _ in range(T)]).astype(np.int32)
    s, e, npp = sba.moe_align_block_size(torch.from_numpy(ids).to(gpu), tile, E)
    rs, re, rn = awq_ref.moe_align(ids, E, tile)
    n = T * topk
    assert int(npp.item()) == rn
    s, e = s.cpu().numpy(), e.cpu().numpy()
    assert np.array_equal(s[:rn], rs)
    assert np.array_equal(e[:rn // tile], re)
    assert np.all(s[rn:] == n) and np.all(e[rn // tile:] == -1)


def _moe_arrays(fx):
    w13 = (fx["w13_qweight"], fx["w13_scales"], fx["w13_qzeros"])
    w2 = (fx["w2_qweight"], fx["w2_scales"], fx["w2_qzeros"])
    return w13, w2


def _run_moe(sba, dev, x, logits, w13, w2, topk):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    y = sba.fused_moe_awq(t(x), tuple(t(a) for a in w13), tuple(t(a) for a in w2), t(logits), topk, True)
    torch.cuda.synchronize()
    return y.cpu().numpy()


def test_moe_fixture(sba, gpu):
    fx = np.load(os.path.join(GOLDEN, "awq_moe_small.npz"))
    w13, w2 = _moe_arrays(fx)
    y = _run_moe(sba, gpu, fx["x"], fx["logits"], w13, w2, int(fx["topk"]))
    err = awq_ref.rel_frobenius(y, fx["y"])
    print(f"[moe fixture] rel_fro={err:.2e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("bs", [16, 32])
def test_moe_grouped_gemm_block_sizes(sba, gpu, bs):
    """The grouped GEMM alone, 16- and 32-row blocks, against per-slot oracle products."""
    rng = np.random.default_rng(40 + bs)
    T, E, topk, K, N, G = 37, 8, 2, 256, 264 if bs == 16 else 256, 128
    w = rng.integers(0, 16, (E, K, N))
    z = rng.integers(0, 16, (E, K // G, N))
    s = (rng.random((E, K // G, N)) * 0.019 + 0.001).astype(np.float16)
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    x = rng.normal(0, 1, (T, K)).astype(np.float16)
    ids = np.stack([rng.choice(E, size=topk, replace=False) for _ in range(T)]).astype(np.int32)
    tw = rng.random((T, topk)).astype(np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    sid, eid, npp = sba.moe_align_block_size(t(ids), bs, E)
    y = sba.moe_awq_gemm(t(x), t(qw), t(s), t(qz), sid, eid, npp, T * topk, topk, topk_weights=t(tw),
                         split_k=2, block_size=bs).cpu().numpy()
    ref = np.zeros((T * topk, N))
    for tok in range(T):
        for slot in range(topk):
            e = ids[tok, slot]
            ref[tok * topk + slot] = awq_ref.gemm_wide(x[tok:tok + 1], qw[e], s[e], qz[e], G)[0] * tw[tok, slot]
    err = awq_ref.rel_frobenius(y, ref)
    print(f"[moe grouped gemm bs={bs}] rel_fro={err:.2e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("T,E,topk,K,N,G", [
    (37, 8, 2, 256, 264, 128),      # ragged last word column, an odd number of 128-column blocks
    (300, 6, 2, 768, 512, 128),     # several blocks per expert, three chunks per wave
    (97, 5, 1, 512, 384, 64),       # top-1, group 64
    (64, 4, 2, 256, 128, 32),       # group 32, a single column block
    (1, 4, 2, 1024, 2048, 128),     # a single token: every block is nearly all padding
])
@pytest.mark.parametrize("variant", [None, 4096, 1 << 27])
def test_moe_grouped_gemm_32_row_forms(sba, gpu, T, E, topk, K, N, G, variant):
    """32-row sorted-token blocks without a K split: one packed word per lane with the weight ring in
    LDS (default), the same with the ring in registers (4096), and the two-words-per-lane form
    (1 << 27, N % 16 == 0 only), against per-slot oracle products."""
    if variant == (1 << 27) and N % 16 != 0:
        pytest.skip("two words per lane need N % 16 == 0")
    rng = np.random.default_rng(T + K + N)
    w = rng.integers(0, 16, (E, K, N))
    z = rng.integers(0, 16, (E, K // G, N))
    s = (rng.random((E, K // G, N)) * 0.019 + 0.001).astype(np.float16)
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    x = rng.normal(0, 1, (T, K)).astype(np.float16)
    ids = np.stack([rng.choice(E, size=topk, replace=False) for _ in range(T)]).astype(np.int32)
    tw = rng.random((T, topk)).astype(np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    sid, eid, npp = sba.moe_align_block_size(t(ids), 32, E)
    out = torch.full((T * topk, N), float("nan"), dtype=torch.float16, device=gpu)
    y = sba.moe_awq_gemm(t(x), t(qw), t(s), t(qz), sid, eid, npp, T * topk, topk, topk_weights=t(tw),
                         block_size=32, out=out, _dev_variant=variant).cpu().numpy()
    assert np.all(np.isfinite(y))            # every slot row written
    ref = np.zeros((T * topk, N))
    for e in range(E):
        tok, slot = np.nonzero(ids == e)
        if tok.size:
            ref[tok * topk + slot] = awq_ref.gemm_wide(x[tok], qw[e], s[e], qz[e], G) * tw[tok, slot][:, None]
    err = awq_ref.rel_frobenius(y, ref)
    print(f"[moe grouped 32-row T={T} K={K} N={N} G={G} variant={variant}] rel_fro={err:.2e}", flush=True)
    assert err <= TOL
    # one X row per slot (the second expert GEMM's addressing), no routing weight
    xs = rng.normal(0, 1, (T * topk, K)).astype(np.float16)
    y2 = sba.moe_awq_gemm(t(xs), t(qw), t(s), t(qz), sid, eid, npp, T * topk, 1, block_size=32,
                          _dev_variant=variant).cpu().numpy()
    ref2 = np.zeros((T * topk, N))
    flat = ids.reshape(-1)
    for e in range(E):
        rows = np.nonzero(flat == e)[0]
        if rows.size:
            ref2[rows] = awq_ref.gemm_wide(xs[rows], qw[e], s[e], qz[e], G)
    assert awq_ref.rel_frobenius(y2, ref2) <= TOL


@pytest.mark.parametrize("bs,T,E,topk,K,N,G", [
    (64, 300, 6, 2, 256, 264, 128),     # ragged last column tile, ragged last blocks
    (128, 300, 6, 2, 256, 264, 128),
    (256, 300, 6, 2, 256, 264, 128),
    (64, 97, 5, 1, 384, 512, 64),       # top-1, group 64, K = 6 k-tiles
    (128, 1, 4, 2, 128, 256, 32),       # a single token: every block is nearly all padding
    (128, 700, 3, 3, 640, 1024, 128),   # several blocks per expert
])
def test_moe_grouped_gemm_mfma_blocks(sba, gpu, bs, T, E, topk, K, N, G):
    """The grouped GEMM over 64 / 128 / 256-row blocks (the tile kernel's expert-grouped form)
    against per-slot oracle products, with routing weights."""
    rng = np.random.default_rng(bs + T + K)
    w = rng.integers(0, 16, (E, K, N))
    z = rng.integers(0, 16, (E, K // G, N))
    s = (rng.random((E, K // G, N)) * 0.019 + 0.001).astype(np.float16)
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    x = rng.normal(0, 1, (T, K)).astype(np.float16)
    ids = np.stack([rng.choice(E, size=topk, replace=False) for _ in range(T)]).astype(np.int32)
    tw = rng.random((T, topk)).astype(np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    sid, eid, npp = sba.moe_align_block_size(t(ids), bs, E)
    out = torch.full((T * topk, N), float("nan"), dtype=torch.float16, device=gpu)
    y = sba.moe_awq_gemm(t(x), t(qw), t(s), t(qz), sid, eid, npp, T * topk, topk, topk_weights=t(tw),
                         block_size=bs, out=out).cpu().numpy()
    assert np.all(np.isfinite(y))            # every slot row written
    ref = np.zeros((T * topk, N))
    for e in range(E):
        tok, slot = np.nonzero(ids == e)
        if tok.size:
            ref[tok * topk + slot] = awq_ref.gemm_wide(x[tok], qw[e], s[e], qz[e], G) * tw[tok, slot][:, None]
    err = awq_ref.rel_frobenius(y, ref)
    print(f"[moe grouped mfma bs={bs} T={T}] rel_fro={err:.2e}", flush=True)
    assert err <= TOL
    # same ids, no routing weight, one X row per slot (the second expert GEMM's addressing)
    xs = rng.normal(0, 1, (T * topk, K)).astype(np.float16)
    y2 = sba.moe_awq_gemm(t(xs), t(qw), t(s), t(qz), sid, eid, npp, T * topk, 1, block_size=bs).cpu().numpy()
    ref2 = np.zeros((T * topk, N))
    flat = ids.reshape(-1)
    for e in range(E):
        rows = np.nonzero(flat == e)[0]
        if rows.size:
            ref2[rows] = awq_ref.gemm_wide(xs[rows], qw[e], s[e], qz[e], G)
    assert awq_ref.rel_frobenius(y2, ref2) <= TOL


@pytest.mark.parametrize("bs", [64, 128, 256])
def test_moe_grouped_gemm_partly_filled_blocks(sba, gpu, bs):
    """Blocks of the grouped tile kernel run on tiles of as many rows as they hold real slots:
    experts with row counts on both sides of every 64 rows, one expert without rows, one with
    several blocks, against per-expert oracle products."""
    counts = [1, 64, 65, 128, 0, 129, 192, 193, 256, 257, 3 * 256 + 66]
    E, K, N, G = len(counts), 256, 264, 64
    rng = np.random.default_rng(bs)
    w = rng.integers(0, 16, (E, K, N))
    z = rng.integers(0, 16, (E, K // G, N))
    s = (rng.random((E, K // G, N)) * 0.019 + 0.001).astype(np.float16)
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)[:, None]
    T = len(ids)
    x = rng.normal(0, 1, (T, K)).astype(np.float16)
    tw = rng.random((T, 1)).astype(np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    sid, eid, npp = sba.moe_align_block_size(t(ids), bs, E)
    out = torch.full((T, N), float("nan"), dtype=torch.float16, device=gpu)
    y = sba.moe_awq_gemm(t(x), t(qw), t(s), t(qz), sid, eid, npp, T, 1, topk_weights=t(tw), block_size=bs,
                         out=out).cpu().numpy()
    assert np.all(np.isfinite(y))            # every slot row written
    for e in range(E):
        tok = np.nonzero(ids[:, 0] == e)[0]
        if tok.size:
            ref = awq_ref.gemm_wide(x[tok], qw[e], s[e], qz[e], G) * tw[tok]
            assert awq_ref.rel_frobenius(y[tok], ref) <= TOL, e


@pytest.mark.parametrize("bs", [64, 128, 256])
def test_moe_grouped_gemm_partly_filled_blocks_of_any_group(sba, gpu, bs):
    """The same steps of 64 rows in groups that are no power of two (a kernel instantiation of their own)."""
    counts = [64, 65, 0, 128, 129, 192, 193, 256, 1, 256 + 66]
    E, K, N, G = len(counts), 768, 136, 384
    rng = np.random.default_rng(bs)
    w, z = rng.integers(0, 16, (E, K, N)), rng.integers(0, 16, (E, K // G, N))
    s = (rng.random((E, K // G, N)) * 0.019 + 0.001).astype(np.float16)
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)[:, None]
    x = rng.normal(0, 1, (len(ids), K)).astype(np.float16)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    sid, eid, npp = sba.moe_align_block_size(t(ids), bs, E)
    out = torch.full((len(ids), N), float("nan"), dtype=torch.float16, device=gpu)
    y = sba.moe_awq_gemm(t(x), t(qw), t(s), t(qz), sid, eid, npp, len(ids), 1, block_size=bs, out=out).cpu().numpy()
    assert np.all(np.isfinite(y))            # every slot row written
    for e in range(E):
        rows = np.nonzero(ids[:, 0] == e)[0]
        if rows.size:
            assert awq_ref.rel_frobenius(y[rows], awq_ref.gemm_wide(x[rows], qw[e], s[e], qz[e], G)) <= TOL, e


TILE_EDGES = [1, 16, 17, 32, 33, 48, 0, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 177, 241, 257, 300]


@pytest.mark.parametrize("E", [len(TILE_EDGES), 13])     # 16 experts or more: tiles dealt to the XCDs in ranges
@pytest.mark.parametrize("bs,K,N,G", [
    (64, 128, 256, 128), (128, 256, 264, 64), (256, 640, 512, 128), (256, 1280, 288, 128),   # 2 ... 20 stages of 64 k
    (128, 256, 72, 32), (256, 384, 520, 384), (64, 256, 40, 64),      # groups and columns of the general form
    (128, 1280, 264, 32), (256, 1152, 512, 32),                       # ... over more stages than the ring holds
])
def test_moe_grouped_gemm_at_the_tile_edges(sba, gpu, bs, K, N, G, E):
    """The grouped kernel takes the lowest tile, in steps of 16 rows, that holds a block's slots (a block of 256 runs as
    two): experts with slot counts on both sides of every step, against per-expert oracle products."""
    counts = TILE_EDGES[:E] if bs < 256 else TILE_EDGES[-E:]
    rng = np.random.default_rng(bs + K + E)
    w, z = rng.integers(0, 16, (E, K, N)), rng.integers(0, 16, (E, K // G, N))
    s = (rng.random((E, K // G, N)) * 0.019 + 0.001).astype(np.float16)
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)[:, None]
    T = len(ids)
    x = rng.normal(0, 1, (T, K)).astype(np.float16)
    tw = rng.random((T, 1)).astype(np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    sid, eid, npp = sba.moe_align_block_size(t(ids), bs, E)
    out = torch.full((T + 1, N), float("nan"), dtype=torch.float16, device=gpu)
    y = sba.moe_awq_gemm(t(x), t(qw), t(s), t(qz), sid, eid, npp, T, 1, topk_weights=t(tw), block_size=bs, out=out[:T])
    y = y.cpu().numpy()
    assert np.all(np.isfinite(y)) and bool(torch.isnan(out[T]).all())      # every slot row written, none behind them
    for e in range(E):
        tok = np.nonzero(ids[:, 0] == e)[0]
        if tok.size:
            ref = awq_ref.gemm_wide(x[tok], qw[e], s[e], qz[e], G) * tw[tok]
            assert awq_ref.rel_frobenius(y[tok], ref) <= TOL, e


# 16-slot blocks in tiles of up to four; 64, 128, 256; the same with a separate activation kernel (no tiles then)
@pytest.mark.parametrize("variant", [512, 1 << 16, 2 << 16, 3 << 16, 512 | 1024, 2 << 16 | 1024])
@pytest.mark.parametrize("H,I,G,E", [(256, 128, 128, 22), (384, 384, 64, 22), (1152, 256, 128, 13), (128, 640, 64, 13)])
def test_fused_call_on_the_grouped_kernel_at_the_tile_edges(sba, gpu, variant, H, I, G, E):
    """The one-call block with both expert GEMMs on the grouped kernel, the first writing silu(gate) * up itself, over
    experts with slot counts on both sides of every tile step: against dense experts, and bit for bit against itself."""
    counts = TILE_EDGES[:E]
    T = sum(counts)
    c = sba.workloads.make_moe_case(T, H, E, 1, I, G, seed=H + I).to(gpu)
    own = torch.from_numpy(np.random.default_rng(T).permutation(np.repeat(np.arange(E), counts))).to(gpu)
    c.logits.clamp_(-3, 3)
    c.logits[torch.arange(T, device=gpu), own] = 8.0       # top-1 goes there
    run = lambda v: sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 1, True, _dev_variant=v)
    y = run(variant).clone()
    assert torch.equal(y.view(torch.int16), run(variant).view(torch.int16))
    ref = _dense_expert_reference(sba, c, gpu, T, H, E, 1, I)
    plain = run(2048).float()
    for e in range(E):
        r = own == e
        if bool(r.any()):
            assert float((y[r].float() - ref[r]).norm() / ref[r].norm()) <= TOL, e
            assert float((y[r].float() - plain[r]).norm() / plain[r].norm()) <= TOL, e


@pytest.mark.parametrize("G", [64, 128])
def test_tiles_of_16_slot_blocks_are_as_near_to_64_bits_as_single_blocks(sba, gpu, G):
    """16-slot blocks in tiles add their group sums in another order than one by one, and subtract the zero points before the
    product instead of behind it: the result moves by some 2e-4 (the roundings of gate / up, activation and slot row on the way),
    not further from the product in 64 bits."""
    T, H, I, E = 1000, 1024, 512, 16
    c = sba.workloads.make_moe_case(T, H, E, 1, I, G, seed=G).to(gpu)
    own = torch.arange(T, device=gpu) % E
    c.logits.zero_()
    c.logits[torch.arange(T, device=gpu), own] = 8.0
    def exact(q, s, z):
        w = awq_ref.unpack_awq(q.cpu().numpy()).astype(np.float64) - awq_ref.unpack_awq(z.cpu().numpy()).astype(np.float64).repeat(G, 0)
        return torch.from_numpy(w * s.cpu().numpy().astype(np.float64).repeat(G, 0)).to(gpu)
    ref = torch.empty((T, H), dtype=torch.float64, device=gpu)
    for e in range(E):
        gate, up = (c.x[own == e].double() @ exact(*(t[e] for t in c.w13))).chunk(2, dim=-1)
        ref[own == e] = (torch.nn.functional.silu(gate) * up) @ exact(*(t[e] for t in c.w2))
    tiles, single = (sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 1, True, _dev_variant=v).double() for v in (512, 2048))
    assert not torch.equal(tiles, single)
    # 1 %: what the two do not share, about half of either error, moves the norm of a million values' error by 0.1 %
    assert float((tiles - ref).norm()) <= 1.01 * float((single - ref).norm())


@pytest.mark.parametrize("T,H,E,topk,I,G", [(320, 1024, 64, 4, 512, 128), (440, 1024, 64, 4, 512, 64), (400, 2048, 128, 8, 768, 128)])
def test_blocks_of_twenty_slots_per_expert_are_as_near_to_64_bits_in_tiles(sba, gpu, T, H, E, topk, I, G):
    """From 20 to 28 slots per expert, where the call takes its 16-slot blocks in tiles by its own rule: several picks a token, the
    block against exact weights and float64 sums, routed as the kernel routed it, beside the same block on single blocks."""
    from server_benchmark_amd import _lib
    assert _lib.load().awqmi_dev_fused_moe_tiles(T, H, I, E, topk, G, -1) == 1 and 20 <= T * topk / E < 28
    c = sba.workloads.make_moe_case(T, H, E, topk, I, G, seed=T + G).to(gpu)
    w, ids = sba.topk_softmax(c.logits, topk, True)
    def exact(q, s, z):
        v = awq_ref.unpack_awq(q.cpu().numpy()).astype(np.float64) - awq_ref.unpack_awq(z.cpu().numpy()).astype(np.float64).repeat(G, 0)
        return torch.from_numpy(v * s.cpu().numpy().astype(np.float64).repeat(G, 0)).to(gpu)
    ref = torch.zeros((T, H), dtype=torch.float64, device=gpu)
    for e in range(E):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        gate, up = (c.x[tok].double() @ exact(*(t[e] for t in c.w13))).chunk(2, dim=-1)
        o = (torch.nn.functional.silu(gate) * up) @ exact(*(t[e] for t in c.w2))
        ref.index_add_(0, tok, o * w[tok, slot].double()[:, None])
    tiles, single = (sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, _dev_variant=v).double() for v in (-1, 2048))
    assert not torch.equal(tiles, single)
    err = [float((y - ref).norm() / ref.norm()) for y in (tiles, single)]
    print(f"[moe tiles T={T} E={E} G={G}] to 64 bits {err[0]:.5e}, single blocks {err[1]:.5e}", flush=True)
    # 1 %: half of either error is not shared (above); 300 thousand values' norm moves by 0.2 %
    assert err[0] <= 1.01 * err[1]


@pytest.mark.parametrize("T,H,E,topk,I,mfma", [(2048, 2048, 128, 8, 768, False), (1024, 1024, 8, 2, 2048, False),
                                               (4096, 512, 4, 2, 384, False),     # many rows per expert
                                               (640, 256, 4, 1, 1152, False),     # top-1
                                               (8192, 2048, 128, 8, 768, True), (4096, 2048, 64, 6, 1408, True)])
def test_fused_call_on_prefill_batches(sba, gpu, T, H, E, topk, I, mfma):
    """Batches with many slots per expert, where the one-call path takes 16-row blocks, one by one with the
    weight ring in LDS or (first case) in tiles of up to four, or (mfma) 64 / 128 / 256-row blocks of the tile kernel:
    against the dense expert path and against the step-by-step path over 16-row blocks."""
    from server_benchmark_amd import _lib
    assert (_lib.load().awqmi_fused_moe_block_rows(T, H, I, E, topk, 128) >= 64) == mfma
    assert _lib.load().awqmi_dev_fused_moe_tiles(T, H, I, E, topk, 128, -1) == (T == 2048)
    c = sba.workloads.make_moe_case(T, H, E, topk, I, 128, seed=T + I).to(gpu)
    one = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True)
    ref = _dense_expert_reference(sba, c, gpu, T, H, E, topk, I)
    err = float((one.float() - ref).norm() / ref.norm())
    step = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, block_size=16)
    d = float((one.float() - step.float()).norm() / step.float().norm())
    print(f"[moe prefill T={T} E={E}] vs dense experts {err:.2e}, vs 16-row blocks {d:.2e}", flush=True)
    assert err <= TOL and d <= TOL
    assert torch.equal(one, sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True))


@pytest.mark.parametrize("T", [1, 16])
def test_moe_qwen3_shapes_vs_oracle(sba, gpu, T):
    c = sba.workloads.make_moe_case(T, 2048, 128, 8, 768, 128, seed=100 + T)
    x, logits = c.x.numpy(), c.logits.numpy()
    w13 = tuple(a.numpy() for a in c.w13)
    w2 = tuple(a.numpy() for a in c.w2)
    y = _run_moe(sba, gpu, x, logits, w13, w2, 8)
    ids, tw = awq_ref.topk_softmax(logits, 8, True)
    ref = awq_ref.moe_forward(x, w13, w2, ids, tw, 128)
    err = awq_ref.rel_frobenius(y, ref)
    print(f"[moe T={T}] rel_fro={err:.2e} max_abs={np.max(np.abs(y.astype(np.float64) - ref)):.3e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("T", [128, 512])
def test_moe_qwen3_shapes_vs_dense_expert_path(sba, gpu, T):
    """At sizes where the per-token CPU loop is too slow: evaluate every expert densely on the
    GPU with the (bit-exact) dequantize kernel + a library matmul and combine with the routing
    weights; the grouped path must agree."""
    c = sba.workloads.make_moe_case(T, 2048, 128, 8, 768, 128, seed=100 + T).to(gpu)
    y = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)
    w, ids = sba.topk_softmax(c.logits, 8, True)
    ref = torch.zeros((T, 2048), dtype=torch.float32, device=gpu)
    for e in range(128):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        W13 = sba.awq_dequantize(c.w13[0][e], c.w13[1][e], c.w13[2][e]).float()
        W2 = sba.awq_dequantize(c.w2[0][e], c.w2[1][e], c.w2[2][e]).float()
        h = (c.x[tok].float() @ W13).half().float()
        a = (torch.nn.functional.silu(h[:, :768]) * h[:, 768:]).half().float()
        o = ((a @ W2) * w[tok, slot][:, None]).half().float()
        ref.index_add_(0, tok, o)
    err = awq_ref.rel_frobenius(y.cpu().numpy(), ref.cpu().numpy())
    print(f"[moe T={T} vs dense experts] rel_fro={err:.2e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("T", [1, 7, 64])
def test_fused_call_equals_step_by_step(sba, gpu, T):
    """The one-call block and the six separate calls run the same kernels on the same data:
    bit-identical outputs, also on a second call that reuses the workspace."""
    c = sba.workloads.make_moe_case(T, 512, 16, 4, 256, 128, seed=7 + T).to(gpu)
    step = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 4, True, block_size=16)
    for _ in range(2):
        one = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 4, True)
        assert torch.equal(one, step)


def test_fused_call_graph_replay(sba, gpu):
    """Captured once, replayed with eager work in between: every replay equals the eager result."""
    c = sba.workloads.make_moe_case(16, 2048, 128, 8, 768, 128, seed=3).to(gpu)
    eager = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)   # sizes this stream's workspace
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            y = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, eager)
            y.zero_()
            sba.awq_gemm(c.x, c.w13[0][0], c.w13[1][0], c.w13[2][0], 0)   # unrelated eager work
            torch.cuda.synchronize()
    torch.cuda.current_stream().wait_stream(s)


def test_graph_survives_workspace_growth(sba, gpu):
    """A graph captured with a small per-stream workspace must stay valid after a later, larger
    call on the same stream has made the wrapper allocate a bigger one: the outgrown buffer is
    kept alive, so the replay still finds its counters and scratch space."""
    from server_benchmark_amd import ops
    c = sba.workloads.make_moe_case(4, 2048, 128, 8, 768, 128, seed=9).to(gpu)
    eager = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)
        torch.cuda.synchronize()
        small = ops.get_workspace(gpu, 1)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            y = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)
        big = sba.workloads.make_moe_case(3000, 2048, 128, 8, 768, 128, seed=10).to(gpu)
        sba.fused_moe_awq(big.x, big.w13, big.w2, big.logits, 8, True)      # outgrows the workspace
        torch.cuda.synchronize()
        grown = ops.get_workspace(gpu, 1)
        assert grown.data_ptr() != small.data_ptr() and grown.numel() >= 2 * small.numel()
        del small
        filler = torch.full((64 << 20,), 0x5A, dtype=torch.uint8, device=gpu)   # would reuse freed memory
        for _ in range(2):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, eager)
        del filler
    torch.cuda.current_stream().wait_stream(s)


def _dense_expert_reference(sba, c, gpu, T, H, E, topk, I):
    """Every expert evaluated densely with the dequantize kernel + a library matmul."""
    w, ids = sba.topk_softmax(c.logits, topk, True)
    ref = torch.zeros((T, H), dtype=torch.float32, device=gpu)
    for e in range(E):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        W13 = sba.awq_dequantize(c.w13[0][e], c.w13[1][e], c.w13[2][e]).float()
        W2 = sba.awq_dequantize(c.w2[0][e], c.w2[1][e], c.w2[2][e]).float()
        h = (c.x[tok].float() @ W13).half().float()
        a = (torch.nn.functional.silu(h[:, :I]) * h[:, I:]).half().float()
        o = ((a @ W2) * w[tok, slot][:, None]).half().float()
        ref.index_add_(0, tok, o)
    return ref


@pytest.mark.parametrize("T,H,E,topk,I", [
    (8192, 2048, 32, 8, 768),    # more (block, column block) tiles than arrival counters: split-K is switched off
    (300, 384, 60, 3, 128),      # expert count that is no multiple of 64, odd top-k, ragged last blocks
    (40, 256, 8, 1, 384),        # top-1, K of the second GEMM = 3 chunks (no column-block pairing)
    (64, 256, 200, 8, 256),      # most experts idle
])
def test_moe_odd_shapes_vs_dense_expert_path(sba, gpu, T, H, E, topk, I):
    c = sba.workloads.make_moe_case(T, H, E, topk, I, 128, seed=T + E).to(gpu)
    y = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True)
    ref = _dense_expert_reference(sba, c, gpu, T, H, E, topk, I)
    err = float((y.float() - ref).norm() / ref.norm())
    print(f"[moe odd T={T} E={E} topk={topk}] rel_fro={err:.2e}", flush=True)
    assert err <= TOL
    assert torch.equal(y, sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True))
    y16 = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, block_size=16)
    assert float((y16.float() - ref).norm() / ref.norm()) <= TOL


@pytest.mark.parametrize("T", [1, 4, 128, 512])
def test_fused_activation_agrees_with_step_by_step(sba, gpu, T):
    """Block sizes at which the w13 GEMM of the one-call path writes silu(gate) * up itself (T = 1, 4:
    split in K, the last arrivers of a gate block and its up block apply it; 128, 512: gate and up
    block in one workgroup).  Its
    two waves per column block add K in another order than the four of the separate-kernel
    path, so the two agree to fp32 summation order (a few last-bit differences after the fp16
    roundings), not bit for bit; both must meet the tolerance against the dense expert path."""
    c = sba.workloads.make_moe_case(T, 2048, 128, 8, 768, 128, seed=300 + T).to(gpu)
    step = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True, block_size=16)
    one = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True)
    d = float((one.float() - step.float()).norm() / step.float().norm())
    print(f"[moe fused act T={T}] vs step-by-step rel_fro={d:.2e}", flush=True)
    assert d <= 2e-4
    ref = _dense_expert_reference(sba, c, gpu, T, 2048, 128, 8, 768)
    assert float((one.float() - ref).norm() / ref.norm()) <= TOL
    assert torch.equal(one, sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, 8, True))


@pytest.mark.parametrize("T,H,E,topk,I,G", [(256, 2048, 128, 8, 768, 128), (16, 1024, 16, 16, 512, 64),
                                            (64, 512, 8, 2, 256, 32), (300, 2048, 128, 8, 768, 128),
                                            (40, 768, 8, 4, 384, 384)])
def test_lds_weight_ring_is_bit_identical(sba, gpu, T, H, E, topk, I, G):
    """From one full 16-row block per expert on, the expert GEMMs keep their weight ring in LDS
    (filled by direct-to-LDS buffer loads); with that form switched off (development variant
    bit 4096) the block must give the same bits."""
    assert T * topk >= 16 * E
    c = sba.workloads.make_moe_case(T, H, E, topk, I, G, seed=T + 5).to(gpu)
    y = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True).clone()
    y_reg = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, _dev_variant=4096).clone()
    assert torch.equal(y.view(torch.int16), y_reg.view(torch.int16))


@pytest.mark.parametrize("T,E,topk", [(1, 128, 8), (33, 128, 8), (7, 160, 6), (5, 16, 2)])
def test_topk_sigmoid_with_bias(sba, gpu, T, E, topk):
    g = torch.Generator().manual_seed(T * 3 + E)
    logits = torch.randn((T, E), generator=g)
    bias = torch.randn((E,), generator=g) * 0.1
    for renorm, b, scale in ((True, bias, 2.5), (False, None, 1.0), (True, None, 1.0)):
        w, ids = sba.topk_route(logits.to(gpu), topk, renorm, "sigmoid", None if b is None else b.to(gpu), scale)
        rid, rw = awq_ref.topk_sigmoid(logits.numpy(), topk, renorm, None if b is None else b.numpy(), scale)
        assert np.array_equal(ids.cpu().numpy(), rid)
        assert np.allclose(w.cpu().numpy(), rw, rtol=2e-5, atol=1e-8)


def test_moe_block_sigmoid_routing(sba, gpu):
    """The block with sigmoid routing + bias + scaling factor against the oracle's forward with
    the oracle's routing."""
    c = sba.workloads.make_moe_case(12, 256, 16, 4, 128, 128, seed=77)
    bias = (torch.randn((16,), generator=torch.Generator().manual_seed(5)) * 0.1)
    cg = c.to(gpu)
    y = sba.fused_moe_awq(cg.x, cg.w13, cg.w2, cg.logits, 4, True, scoring_func="sigmoid",
                          e_score_correction_bias=bias.to(gpu), routed_scaling_factor=1.5).cpu().numpy()
    ids, tw = awq_ref.topk_sigmoid(c.logits.numpy(), 4, True, bias.numpy(), 1.5)
    ref = awq_ref.moe_forward(c.x.numpy(), tuple(a.numpy() for a in c.w13), tuple(a.numpy() for a in c.w2),
                              ids, tw, 128)
    assert awq_ref.rel_frobenius(y, ref) <= TOL
    # the one-call path above and the step-by-step path run the same kernels on the same routing
    step = sba.fused_moe_awq(cg.x, cg.w13, cg.w2, cg.logits, 4, True, scoring_func="sigmoid",
                             e_score_correction_bias=bias.to(gpu), routed_scaling_factor=1.5, block_size=16)
    assert np.array_equal(step.cpu().numpy(), y)


@pytest.mark.parametrize("T", [64, 3000])
def test_moe_block_sigmoid_routing_larger_batches(sba, gpu, T):
    """Sigmoid-routed block at batch sizes that take the separate routing kernel and, at 3000
    tokens, the multi-workgroup align and larger blocks: against the dense expert path with the
    routing kernel's own ids and weights."""
    H, E, topk, I = 512, 32, 6, 256
    c = sba.workloads.make_moe_case(T, H, E, topk, I, 128, seed=T).to(gpu)
    bias = (torch.randn((E,), generator=torch.Generator().manual_seed(9)) * 0.1).to(gpu)
    y = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, scoring_func="sigmoid",
                          e_score_correction_bias=bias, routed_scaling_factor=2.5)
    w, ids = sba.topk_route(c.logits, topk, True, "sigmoid", bias, 2.5)
    ref = torch.zeros((T, H), dtype=torch.float32, device=gpu)
    for e in range(E):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        W13 = sba.awq_dequantize(c.w13[0][e], c.w13[1][e], c.w13[2][e]).float()
        W2 = sba.awq_dequantize(c.w2[0][e], c.w2[1][e], c.w2[2][e]).float()
        h = (c.x[tok].float() @ W13).half().float()
        a = (torch.nn.functional.silu(h[:, :I]) * h[:, I:]).half().float()
        ref.index_add_(0, tok, ((a @ W2) * w[tok, slot][:, None]).half().float())
    err = float((y.float() - ref).norm() / ref.norm())
    print(f"[moe sigmoid T={T}] rel_fro={err:.2e}", flush=True)
    assert err <= TOL


def test_empty_batches(sba, gpu):
    """No tokens: every operator returns an empty result of the right shape and launches nothing."""
    c = sba.workloads.make_moe_case(4, 256, 8, 2, 128, 128, seed=1).to(gpu)
    y = sba.fused_moe_awq(c.x[:0], c.w13, c.w2, c.logits[:0], 2, True)
    assert tuple(y.shape) == (0, 256) and y.dtype == torch.float16
    y = sba.fused_moe_awq(c.x[:0], c.w13, c.w2, c.logits[:0], 2, True, block_size=16)
    assert tuple(y.shape) == (0, 256)
    lin = sba.workloads.make_linear_case(2, 256, 64, 128, seed=0).to(gpu)
    y = sba.awq_gemm(lin.x[:0], lin.qweight, lin.scales, lin.qzeros, 0)
    assert tuple(y.shape) == (0, 64) and y.dtype == torch.float16


@pytest.mark.parametrize("T,E,topk", [(2048, 128, 8), (2500, 60, 7), (20000, 8, 2)])
def test_fused_call_with_long_slot_lists(sba, gpu, T, E, topk):
    """On long slot lists the one-call path picks, counts and places with several workgroups;
    there too its result must equal the step-by-step path, whose align
    is the single workgroup checked against the oracle above."""
    H, I = 256, 128
    c = sba.workloads.make_moe_case(T, H, E, topk, I, 128, seed=T + E).to(gpu)
    assert T * topk >= 16384
    one = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True)
    from server_benchmark_amd import _lib
    bs = _lib.load().awqmi_fused_moe_block_rows(T, H, I, E, topk, 128)
    step = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, block_size=bs)
    assert torch.equal(one, step)
    assert torch.equal(one, sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True))


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("T,E,topk", [(32, 128, 8), (33, 128, 8), (16, 64, 17), (17, 64, 17), (256, 128, 8), (257, 128, 8),
                                      (2049, 4, 2), (2050, 5, 1), (300, 1024, 17), (2100, 256, 16), (130, 257, 16), (662, 64, 17), (663, 64, 17),
                                      (448, 128, 8), (449, 128, 8)])
def test_routing_in_one_two_and_several_workgroups(sba, gpu, scoring, T, E, topk):
    """Both sides of the rule for the block's routing launches (32 tokens, 16 with a token a wave; 3584 slots, 11264 with a token
    a wave; a last part of one token): the block must equal the step-by-step path, whose top-k and align are checked against the oracle above."""
    c = sba.workloads.make_moe_case(T, 256, E, topk, 128, 128, seed=T + E).to(gpu)
    kw = {}
    if scoring == "sigmoid":
        kw = dict(scoring_func="sigmoid", e_score_correction_bias=torch.linspace(0, 0.1, E, device=gpu))
    from server_benchmark_amd import _lib
    bs = _lib.load().awqmi_fused_moe_block_rows(T, 256, 128, E, topk, 128)
    for _ in range(2):
        one = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, **kw)
        step = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, block_size=bs, **kw)
        assert torch.equal(one, step)


@pytest.mark.parametrize("T,E,topk", [(449, 128, 8), (2049, 4, 2), (3590, 5, 1), (1200, 256, 3), (2100, 256, 16), (8192, 128, 8),
                                      (700, 1024, 17), (3761, 1024, 3), (4097, 257, 4), (16385, 300, 1)])
def test_parts_leave_the_lists_of_one_workgroup(sba, gpu, T, E, topk):
    """The one-call block with its routing in parts and with the align in one workgroup (development variant 16384): picks,
    weights, sorted slots, block owners and padded count in the workspace are the same words, to the end of the lists, whatever the
    workspace held, and the align's are the oracle's."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    H, I, n = 256, 128, T * topk
    assert n > (3584 if E <= 256 and topk <= 16 else 11264)
    c = sba.workloads.make_moe_case(T, H, E, topk, I, 128, seed=T + E).to(gpu)
    bs = lib.awqmi_fused_moe_block_rows(T, H, I, E, topk, 128)
    need = lib.awqmi_fused_moe_workspace_bytes(T, H, I, E, topk)
    up = lambda v: (v + 255) // 256 * 256
    cap = lib.awqmi_moe_align_capacity(n, E, bs)
    start = up(max(lib.awqmi_moe_gemm_workspace_bytes(n, E, H, 2 * I, 0, bs), lib.awqmi_moe_gemm_workspace_bytes(n, E, I, H, 0, bs))) // 4
    words = [n, n, cap, cap // bs, 1]                  # ids, weights, sorted slots, block owners, padded count
    lists, outs = [], []
    for variant, fill in ((-1, 0x55), (16384, 0x33)):
        ws = torch.full((need,), fill, dtype=torch.uint8, device=gpu)
        ws[:65536] = 0                                 # arrival counters
        y = torch.empty((T, H), dtype=torch.float16, device=gpu)
        st = lib.awqmi_dev_fused_moe_routed_f16(
            c.x.data_ptr(), c.logits.data_ptr(), 0, *(t.data_ptr() for t in (*c.w13, *c.w2)), y.data_ptr(), T, H, I, E, topk, 128, 0, 1,
            1.0, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream, variant)
        assert st == 0
        w, at, got = ws[:need // 4 * 4].view(torch.int32), start, []
        for k in words:
            got.append(w[at:at + k].cpu())
            at += up(4 * k) // 4
        lists.append(got)
        outs.append(y)
    for a, b in zip(*lists):
        assert torch.equal(a, b)
    rs, re, rn = awq_ref.moe_align(lists[0][0].numpy().reshape(T, topk), E, bs)
    s, e = lists[0][2].numpy(), lists[0][3].numpy()
    assert int(lists[0][4]) == rn and np.array_equal(s[:rn], rs) and np.array_equal(e[:rn // bs], re)
    assert np.all(s[rn:] == n) and np.all(e[rn // bs:] == -1)
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("T,H,E,topk,I", [(1, 2048, 128, 8, 768), (2, 2048, 128, 8, 768), (3, 2048, 128, 8, 768),
                                          (4, 2048, 128, 8, 768), (4, 512, 64, 6, 256), (1, 256, 8, 1, 128),
                                          (3, 1024, 16, 10, 512), (4, 256, 4, 4, 128), (2, 384, 100, 16, 128),
                                          (4, 512, 128, 16, 256), (2, 256, 160, 8, 128), (4, 256, 256, 8, 128)])
def test_routing_folded_into_the_first_expert_gemm(sba, gpu, scoring, T, H, E, topk, I):
    """Blocks of a few tokens (here one to four, up to 64 slots and 256 experts) have no routing launch: the first
    expert GEMM works the routing out in every workgroup.  The result must have the bits of the
    block with the routing launched on its own (development variant bit 1 << 24), also with
    duplicate experts across tokens (few experts, large top-k), and must match the oracle's
    forward with the oracle's routing."""
    c = sba.workloads.make_moe_case(T, H, E, topk, I, 128, seed=11 * T + E)
    cg = c.to(gpu)
    kw = {}
    bias = None
    if scoring == "sigmoid":
        bias = torch.randn((E,), generator=torch.Generator().manual_seed(E)) * 0.1
        kw = dict(scoring_func="sigmoid", e_score_correction_bias=bias.to(gpu), routed_scaling_factor=1.25)
    y = sba.fused_moe_awq(cg.x, cg.w13, cg.w2, cg.logits, topk, True, **kw).clone()
    y_sep = sba.fused_moe_awq(cg.x, cg.w13, cg.w2, cg.logits, topk, True, _dev_variant=1 << 24, **kw).clone()
    assert torch.equal(y.view(torch.int16), y_sep.view(torch.int16))
    if scoring == "sigmoid":
        ids, tw = awq_ref.topk_sigmoid(c.logits.numpy(), topk, True, bias.numpy(), 1.25)
    else:
        ids, tw = awq_ref.topk_softmax(c.logits.numpy(), topk, True)
    ref = awq_ref.moe_forward(c.x.numpy(), tuple(a.numpy() for a in c.w13), tuple(a.numpy() for a in c.w2),
                              ids, tw, 128)
    assert awq_ref.rel_frobenius(y.cpu().numpy(), ref) <= TOL
    # a second call on the same workspace, fewer tokens: nothing of the first call's lists is read
    if T > 1:
        y1 = sba.fused_moe_awq(cg.x[:1].contiguous(), cg.w13, cg.w2, cg.logits[:1].contiguous(), topk, True, **kw)
        y1_sep = sba.fused_moe_awq(cg.x[:1].contiguous(), cg.w13, cg.w2, cg.logits[:1].contiguous(), topk, True,
                                   _dev_variant=1 << 24, **kw)
        assert torch.equal(y1.view(torch.int16), y1_sep.view(torch.int16))


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("T,E,topk", [(5, 128, 8), (8, 128, 8), (8, 4, 4), (7, 256, 9), (8, 33, 8), (5, 16, 12), (3, 64, 16), (9, 128, 7), (10, 128, 7),
                                      (16, 4, 4), (16, 8, 2), (13, 256, 4), (17, 64, 2)])
def test_routing_folded_for_five_to_sixteen_tokens(sba, gpu, scoring, T, E, topk):
    """Up to four waves with four tokens each, up to 64 slots, experts in the first and the last word of the mask; 70 slots, 17
    tokens and a full block for every expert (16 tokens on four) are past the lines.  The bits of the separately routed block."""
    from server_benchmark_amd import _lib
    assert _lib.load().awqmi_dev_fused_moe_folds(T, 512, 256, E, topk, 128, -1) == ((T, E, topk) not in ((10, 128, 7), (16, 4, 4), (17, 64, 2)))
    c = sba.workloads.make_moe_case(T, 512, E, topk, 256, 128, seed=5 * T + E).to(gpu)
    kw = {}
    if scoring == "sigmoid":
        kw = dict(scoring_func="sigmoid", e_score_correction_bias=torch.linspace(0, 0.1, E, device=gpu), routed_scaling_factor=1.25)
    y = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, **kw).clone()
    y_sep = sba.fused_moe_awq(c.x, c.w13, c.w2, c.logits, topk, True, _dev_variant=1 << 24, **kw)
    assert torch.equal(y.view(torch.int16), y_sep.view(torch.int16))


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("T,E,topk,busy", [(16, 8, 4, 0), (16, 8, 4, 7), (9, 64, 2, 63), (16, 64, 2, 0), (13, 33, 4, 32), (16, 256, 4, 255),
                                           (12, 128, 5, 31), (16, 16, 1, 15), (16, 64, 4, 40)])
def test_folded_routing_fills_a_block_to_its_last_row(sba, gpu, scoring, T, E, topk, busy):
    """One expert -- the first, the last, one at a word's edge of the mask -- is picked by all of 9 to 16 tokens, so that its block
    has that many rows: the bits of the separately routed block, and the oracle's result."""
    from server_benchmark_amd import _lib
    assert _lib.load().awqmi_dev_fused_moe_folds(T, 512, 256, E, topk, 128, -1) == 1
    c = sba.workloads.make_moe_case(T, 512, E, topk, 256, 128, seed=3 * T + E + busy)
    c.logits[:, busy] = c.logits.max(dim=1).values + torch.linspace(-0.01, 0.4, T)       # first pick, or (first token) second
    kw = {}
    if scoring == "sigmoid":
        kw = dict(scoring_func="sigmoid", routed_scaling_factor=1.25)
        ids, tw = awq_ref.topk_sigmoid(c.logits.numpy(), topk, True, None, 1.25)
    else:
        ids, tw = awq_ref.topk_softmax(c.logits.numpy(), topk, True)
    assert 9 <= (np.asarray(ids) == busy).sum() >= T - (topk == 1)
    d = c.to(gpu)
    y = sba.fused_moe_awq(d.x, d.w13, d.w2, d.logits, topk, True, **kw).clone()
    y_sep = sba.fused_moe_awq(d.x, d.w13, d.w2, d.logits, topk, True, _dev_variant=1 << 24, **kw)
    assert torch.equal(y.view(torch.int16), y_sep.view(torch.int16))
    ref = awq_ref.moe_forward(c.x.numpy(), tuple(a.numpy() for a in c.w13), tuple(a.numpy() for a in c.w2), ids, tw, 128)
    assert awq_ref.rel_frobenius(y.cpu().numpy(), ref) <= TOL


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("T,E,topk", [(1, 17, 17), (1, 64, 64), (2, 65, 32), (3, 128, 21), (2, 129, 17), (3, 256, 20)])
def test_routing_folded_with_more_than_sixteen_picks(sba, gpu, scoring, T, E, topk):
    """A token a wave, up to three tokens, experts on both sides of one, two and four a lane: the bits of the separately routed block,
    and the oracle's result."""
    from server_benchmark_amd import _lib
    assert _lib.load().awqmi_dev_fused_moe_folds(T, 512, 256, E, topk, 128, -1) == 1
    c = sba.workloads.make_moe_case(T, 512, E, topk, 256, 128, seed=5 * T + E)
    d = c.to(gpu)
    kw = {}
    if scoring == "sigmoid":
        kw = dict(scoring_func="sigmoid", e_score_correction_bias=torch.linspace(0, 0.1, E, device=gpu), routed_scaling_factor=1.25)
        ids, tw = awq_ref.topk_sigmoid(c.logits.numpy(), topk, True, np.linspace(0, 0.1, E, dtype=np.float32), 1.25)
    else:
        ids, tw = awq_ref.topk_softmax(c.logits.numpy(), topk, True)
    y = sba.fused_moe_awq(d.x, d.w13, d.w2, d.logits, topk, True, **kw).clone()
    y_sep = sba.fused_moe_awq(d.x, d.w13, d.w2, d.logits, topk, True, _dev_variant=1 << 24, **kw)
    assert torch.equal(y.view(torch.int16), y_sep.view(torch.int16))
    ref = awq_ref.moe_forward(c.x.numpy(), tuple(a.numpy() for a in c.w13), tuple(a.numpy() for a in c.w2), ids, tw, 128)
    assert awq_ref.rel_frobenius(y.cpu().numpy(), ref) <= TOL


def test_folded_routing_with_nan_logits(sba, gpu):
    """A NaN logit in a folded-routing block: ids stay in range (the block runs, every slot row is
    written) and the output equals the separately routed block's, NaNs included."""
    c = sba.workloads.make_moe_case(2, 512, 16, 4, 256, 128, seed=3).to(gpu)
    lg = c.logits.clone()
    lg[0, 3] = float("nan")
    lg[1, :] = float("nan")
    y = sba.fused_moe_awq(c.x, c.w13, c.w2, lg, 4, True).clone()
    y_sep = sba.fused_moe_awq(c.x, c.w13, c.w2, lg, 4, True, _dev_variant=1 << 24).clone()
    assert torch.equal(y.view(torch.int16), y_sep.view(torch.int16))
