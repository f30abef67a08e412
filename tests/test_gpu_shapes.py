"""Kernels chosen by a rule on sizes, at the sizes where the rule or the tiling can go wrong, against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle as orc
from gpu_util import oracle_weights, qspec, rel_err, to_np
from strixite_amd import moe

pytestmark = pytest.mark.gpu
DEV = "cuda"


def say(*a):
    print("[shapes]", *a, flush=True)


def _bf16(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(DEV).view(torch.bfloat16)


def _weight(bits, N, K, G, seed):
    q, s, m = orc.gen_q(bits, orc.tensor_key(seed, "gu_q"), orc.tensor_key(seed, "gu_s"), N, K, G)
    return moe.QWeight.from_host(bits, q, s, m, N, K, G)


# the served model's K (gate_up 2560: ten streaming waves; down 640: five groups a row, the swizzle of odd group counts)
# at one token, at the most tokens of the decode form, and gathered above it; one slot has an invalid id
# (and each other count of waves and of groups a row that the two kernels take)
@pytest.mark.parametrize("M,A,E,H,I", [(1, 3, 8, 2560, 640), (16, 4, 24, 2560, 640), (17, 4, 9, 2560, 640),
                                       (90, 3, 5, 2560, 640), (5, 3, 9, 2304, 256), (70, 3, 6, 2304, 384),
                                       (7, 4, 9, 2816, 768), (60, 2, 7, 2816, 896), (16, 3, 8, 2048, 1024),
                                       (75, 4, 6, 3072, 1024)])
def test_streamed_experts_at_the_served_widths(M, A, E, H, I):
    say("streamed experts", M, A, E, H, I)
    gu, dn = _weight(4, E * 2 * I, H, 128, 31), _weight(4, E * H, I, 128, 32)
    x = orc.gen_bf16_normal(orc.tensor_key(8, "x"), 1.0, (M, H))
    ids = np.stack([np.random.default_rng(500 + m).permutation(E)[:A] for m in range(M)]).astype(np.int32)
    ids[M // 2, A - 1] = E
    tid = torch.from_numpy(ids).to(DEV)
    ws, _ = moe.moe_group_routes(tid, E)
    ex = moe.MOE_MATH_WMMA_BF16
    h = to_np(moe.experts_gather_grouped_swiglu(_bf16(x), gu, E, ws, M, A, math=ex))
    bad = np.array([M // 2 * A + A - 1])
    good = np.setdiff1d(np.arange(M * A), bad)
    assert np.all(np.isnan(orc.bf16_to_f32(h[bad]))) and not np.isnan(orc.bf16_to_f32(h[good])).any()
    ok_ids = np.where(ids >= E, 0, ids).astype(np.int32)
    b, q, s, m, G = qspec(gu)
    href = orc.experts_gate_up_swiglu(x, orc.qview(b, q, s, m, gu.N, H, G), E, ok_ids)
    assert rel_err(h[good], href[good]) < 1e-2  # h is BF16: one rounding apart, 2^-8 of a value
    hz = h.copy()
    hz[bad] = 0
    pt = torch.full((M * A, H), 7.0, dtype=torch.float32, device=DEV)
    coef = torch.full((M, A), 0.25, device=DEV)
    moe.experts_combine_grouped(_bf16(hz), dn, E, tid, coef, ws, M, A, partial=pt, math=ex)
    p = pt.cpu().numpy()
    assert np.all(np.isnan(p[bad]))
    b, q, s, m, G = qspec(dn)
    pref = orc.experts_down(hz, orc.qview(b, q, s, m, dn.N, I, G), E, ok_ids)
    assert rel_err(p[good], pref[good]) < 1e-4  # FP32 sums of 640 products in another order


def _w64(w: moe.QWeight) -> np.ndarray:
    from oracle import hc

    return hc.weights64(w.bits, to_np(w.q), to_np(w.scale), to_np(w.minv), w.N, w.K, w.G)


def _rel64(got: torch.Tensor, ref: np.ndarray) -> float:
    return float(np.abs(got.double().cpu().numpy() - ref).max() / np.abs(ref).max())


# exact-weight 16-row tiles with FP32 activations: one step of K, K split over 4 and 8 waves, a ragged column end
# (I = 24: half a tile of columns), rows past the tiles, each K step length
@pytest.mark.parametrize("bits,G,K,I", [(4, 128, 128, 24), (4, 128, 4096, 16), (4, 64, 576, 40), (4, 32, 1024, 24),
                                        (8, 64, 448, 24), (8, 128, 2048, 32), (8, 32, 96, 8)])
def test_fp32_activation_tiles(bits, G, K, I):
    say("fp32 tiles", bits, G, K, I)
    M, A, E = 19, 2, 3
    gu = _weight(bits, E * 2 * I, K, G, 41)
    g64 = _w64(gu)
    x = torch.from_numpy(np.random.default_rng(K).standard_normal((M, K)).astype(np.float32)).to(DEV)
    X = x.double().cpu().numpy()
    ids = np.stack([np.random.default_rng(m).permutation(E)[:A] for m in range(M)]).astype(np.int32)
    tid = torch.from_numpy(ids).to(DEV)
    ws, _ = moe.moe_group_routes(tid, E)
    ref = np.stack([X[s // A] @ g64[e * 2 * I:(e + 1) * 2 * I].T for s, e in enumerate(ids.ravel())])
    href = ref[:, :I] / (1 + np.exp(-ref[:, :I])) * ref[:, I:]
    h = moe.experts_gather_grouped_swiglu(x, gu, E, ws, M, A)
    # every product is exact, so the error is that of FP32 sums of up to 4096 terms whose partial sums reach a few
    # times the result (code offsets): ~sqrt(4096) 2^-24 x 4
    assert _rel64(h, href) < 2e-5
    if bits == 4:
        assert _rel64(moe.experts_gather_grouped(x, gu, E, ws, M, A), ref) < 2e-5
        assert torch.equal(moe.experts_gather(x, gu, E, tid, moe.zero_err(), swiglu=True), h)
    lin = moe.linear_q4 if bits == 4 else moe.linear_q8
    d64 = X @ g64.T
    assert _rel64(lin(x, gu, out_dtype=torch.float32), d64) < 2e-5


def test_fp32_router_rows_match_bf16_bits():
    say("fp32 router")
    # FP32 x holding BF16 values: the canonical order's bits, with token counts around the four-token groups, chunk
    # counts that leave lanes without a last chunk, and rows that are not 16-byte aligned
    for M, N, K in [(1, 33, 2560), (2, 5, 520), (5, 17, 1000), (9, 4, 1003), (130, 65, 1003)]:
        rng = np.random.default_rng(M)
        x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(DEV).to(torch.bfloat16)
        w = torch.from_numpy(rng.standard_normal((N, K)).astype(np.float32)).to(DEV).to(torch.bfloat16)
        assert torch.equal(moe.linear_bf16w(x.float(), w), moe.linear_bf16w(x, w)), (M, N, K)


# dense BF16 on either side of the tiles' and the GEMM's sizes, with a remainder of the 16-token tiles
@pytest.mark.parametrize("bits,G,M,N,K", [(8, 64, 17, 1040, 3072), (4, 128, 111, 96, 512), (8, 64, 113, 4096, 2048),
                                          (4, 64, 300, 1024, 2048), (8, 32, 1, 16, 96),
                                          # groups of 32 past the tiles' outputs: the stream kernel, up to K 2048
                                          (4, 32, 555, 528, 512), (8, 32, 421, 992, 1024), (4, 32, 131, 3088, 2048),
                                          (8, 32, 131, 3088, 2080)])
def test_dense_tiles_and_gemm(bits, G, M, N, K):
    say("dense", bits, G, M, N, K)
    w = _weight(bits, N, K, G, 51)
    x = _bf16(orc.gen_bf16_normal(orc.tensor_key(9, "x"), 1.0, (M, K)))
    ref = x.double().cpu().numpy() @ _w64(w).T
    lin = moe.linear_q4 if bits == 4 else moe.linear_q8
    assert _rel64(lin(x, w, out_dtype=torch.float32), ref) < 1e-4  # FP32 sums; the GEMM's Q4 codes carry an offset of 128
    assert _rel64(lin(x, w), ref) < 2.0 ** -8  # one BF16 rounding


# each kernel that dense_plan.hpp chooses from, at ragged tokens and columns: the stream kernel of each format and group size
# past the tiles' outputs, the GEMM (Q4 and Q8, groups of one and two K steps, its tokens' and columns' remainders)
@pytest.mark.parametrize("bits,G,M,N,K", [(8, 64, 85, 4112, 1024), (4, 64, 113, 4096, 1024), (8, 128, 77, 4112, 2048),
                                          (4, 128, 100, 4112, 2048), (4, 64, 70, 8208, 1024), (4, 64, 333, 2064, 1088),
                                          (4, 128, 300, 4112, 1024), (8, 64, 700, 1040, 1088), (8, 128, 400, 2064, 2176)])
def test_dense_stream_and_gemm(bits, G, M, N, K):
    say("dense plan", bits, G, M, N, K)
    w = _weight(bits, N, K, G, 52)
    x = _bf16(orc.gen_bf16_normal(orc.tensor_key(14, "x"), 1.0, (M, K)))
    rows = np.unique(np.concatenate([np.arange(min(M, 20)), np.arange(max(0, M - 20), M)]))
    ref = x.double().cpu().numpy()[rows] @ _w64(w).T
    lin = moe.linear_q4 if bits == 4 else moe.linear_q8
    assert _rel64(lin(x, w, out_dtype=torch.float32)[rows], ref) < 1e-4  # FP32 sums; Q4 codes carry an offset of 128
    assert _rel64(lin(x, w)[rows], ref) < 2.0 ** -8  # one BF16 rounding


# the exact GEMM's blocks dealt to the XCDs in runs: item counts around multiples of 8, one bucket of all the slots,
# an empty one, ragged columns, and a slot with an invalid id
@pytest.mark.parametrize("bits,M,A,E,H,I", [(8, 1090, 1, 1, 128, 128), (8, 520, 2, 3, 192, 144),
                                            (4, 400, 3, 6, 128, 64), (8, 610, 2, 5, 320, 272)])
def test_exact_gemm_items(bits, M, A, E, H, I):
    say("exact gemm", bits, M, A, E, H, I)
    gu, dn = _weight(bits, E * 2 * I, H, 64, 71), _weight(bits, E * H, I // 64 * 64, 64, 72)
    K = dn.K
    x = _bf16(orc.gen_bf16_normal(orc.tensor_key(10, "x"), 1.0, (M, H)))
    h = _bf16(orc.gen_bf16_normal(orc.tensor_key(11, "x"), 1.0, (M * A, K)))
    ids = np.random.default_rng(M).integers(0, max(1, E - 1), size=(M, A)).astype(np.int32)  # the last expert: no slot
    ids[M // 2, A - 1] = E
    tid = torch.from_numpy(ids).to(DEV)
    ws, _ = moe.moe_group_routes(tid, E)
    ex = moe.MOE_MATH_WMMA_BF16
    got = moe.experts_gather_grouped_swiglu(x, gu, E, ws, M, A, math=ex)
    pt = torch.full((M * A, H), 7.0, dtype=torch.float32, device=DEV)
    moe.experts_combine_grouped(h, dn, E, tid, torch.ones((M, A), device=DEV), ws, M, A, partial=pt, math=ex)
    flat = ids.ravel()
    good, bad = np.flatnonzero(flat < E), np.flatnonzero(flat >= E)
    X, Hd, g64, d64 = x.double().cpu().numpy(), h.double().cpu().numpy(), _w64(gu), _w64(dn)
    z = np.stack([X[s // A] @ g64[flat[s] * 2 * I:(flat[s] + 1) * 2 * I].T for s in good])
    p = np.stack([Hd[s] @ d64[flat[s] * H:(flat[s] + 1) * H].T for s in good])
    assert _rel64(got[good], z[:, :I] / (1 + np.exp(-z[:, :I])) * z[:, I:]) < 2.0 ** -8  # one BF16 rounding
    assert _rel64(pt[good], p) < 1e-4  # FP32 sums; Q4 codes carry an offset of 128
    assert torch.isnan(got[bad].float()).all() and torch.isnan(pt[bad]).all()


# the down mix's kernels at the ends of their ranges: lane dots of 2 and 3 tokens and a row remainder, split-K tiles of
# each size (blocks of 16 x 16, 16 x 32, 32 x 32, 32 x 64) with 64- and 32-code steps and streams of a half group, a
# stream too wide for the split's LDS, FP32 lane dots
@pytest.mark.parametrize("bits,G,act,T,d,r,inject", [
    (4, 64, "bf16", 2, 160, 33, False), (8, 32, "bf16", 3, 96, 35, True), (4, 64, "bf16", 33, 160, 20, True),
    (4, 128, "bf16", 49, 320, 64, False), (8, 64, "bf16", 257, 128, 320, True), (4, 32, "bf16", 400, 96, 320, True),
    (4, 64, "bf16", 705, 128, 320, True), (8, 64, "bf16", 1500, 64, 320, False), (4, 32, "bf16", 40, 65536, 8, False),
    (4, 64, "f32", 33, 160, 20, True), (8, 64, "f32", 439, 128, 9, False),
    # FP32 staged tiles, either format and each group size: ragged rows and tokens, one and three stages a stream
    (4, 64, "f32", 500, 128, 1020, True), (8, 64, "f32", 449, 384, 700, False), (4, 32, "f32", 300, 384, 1001, True),
    (8, 128, "f32", 1001, 128, 321, False),
    # BF16 streams too wide for the split-K tiles' LDS, at a token count whose lane dots would cost more than the tiles
    (4, 32, "bf16", 1000, 5120, 316, True),
    # BF16 staged tiles: K in halves of one and of six stages with each group size, one half past the CUs, Q8
    (4, 32, "bf16", 1500, 128, 400, True), (4, 64, "bf16", 1200, 384, 385, False), (4, 128, "bf16", 1500, 128, 400, True),
    (4, 64, "bf16", 1601, 128, 1021, False), (4, 128, "bf16", 1601, 384, 1001, True), (8, 32, "bf16", 1500, 128, 400, True),
    (8, 64, "bf16", 1200, 384, 385, False), (8, 128, "bf16", 1500, 128, 401, True)])
def test_mix_down_kernels(bits, G, act, T, d, r, inject):
    from oracle import hc

    say("mix down", bits, G, act, T, d, r, inject)
    dt = torch.bfloat16 if act == "bf16" else torch.float32
    x = torch.from_numpy(np.random.default_rng(T).standard_normal((T, 4 * d)).astype(np.float32)).to(DEV).to(dt)
    w = _weight(bits, r + (4 if inject else 0), 4 * d, G, 61)
    h, w_in, inv = moe.hc_mix_down(x, w, r, inject, 1e-6)
    rows = np.unique(np.concatenate([np.arange(min(T, 40)), np.arange(max(0, T - 40), T)]))
    hr, wir, invr = hc.hc_mix_down(x.double().cpu().numpy()[rows], _w64(w), d, r, inject, 1e-6)
    # exact products, FP32 sums of 4 d terms of mean zero (codes about the middle of their range): a few 2^-24 sqrt(4 d); the
    # staged tiles' Q4 codes carry an offset of 128: 4e-6 at these widths
    assert _rel64(inv[rows], invr) < 2e-6
    assert _rel64(h[rows], hr) < 1e-5
    if inject:
        assert _rel64(w_in[rows], wir) < 1e-5


# the one-block packing past 1024 slots: around its waves' whole steps, its largest, and the sizes beyond
@pytest.mark.parametrize("M,A,E", [(103, 10, 512), (205, 5, 64), (373, 11, 513), (600, 10, 1023), (6144, 1, 7),
                                   (6145, 1, 7)])
def test_group_routes_one_block_sizes(M, A, E):
    say("packing", M, A, E)
    rng = np.random.default_rng(M)
    ids = rng.integers(0, E, (M, A)).astype(np.int32)
    ids[M // 3, 0], ids[M - 1, A - 1] = -1, E
    ws, err = moe.moe_group_routes(torch.from_numpy(ids).to(DEV), E)
    t = moe.route_tables(ws, M, A, E)
    b = np.where((ids < 0) | (ids >= E), E, ids).ravel()
    counts = np.bincount(b, minlength=E + 1)
    assert np.array_equal(t["offsets"].cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
    assert np.array_equal(t["slots"].cpu().numpy(), np.argsort(b, kind="stable"))
    assert int(t["n_tiles"]) == int(((counts + 15) // 16).sum())
    assert err.cpu().numpy().tolist() == [1, -1, M // 3 * A]


@pytest.mark.parametrize("shared,bits,H,I,E,k", [(True, 4, 512, 256, 32, 4), ("stacked", 4, 2560, 640, 24, 10),
                                                 (False, 8, 512, 128, 64, 8)])
def test_one_token_layer_matches_two(shared, bits, H, I, E, k):
    say("one token", shared, bits, H, I, E, k)
    layer = moe.MoeLayer.synth(H, E, k, I, seed=7, routed_bits=bits, shared=shared)
    x = moe.synth_bf16_normal(7, "x", 0, (2, H), 1.0)
    one, two = layer.forward(x[:1].contiguous()), layer.forward(x)
    assert torch.equal(one["ids"], two["ids"][:1]) and torch.equal(one["coef"], two["coef"][:1])
    y1, y2 = one["y"].double().cpu().numpy(), two["y"][:1].double().cpu().numpy()
    assert np.abs(y1 - y2).max() <= 2.0 ** -7 * np.abs(y2).max()  # one BF16 rounding of each
    # a non-finite logit: invalid ids, NaN rows, both error words
    lg = torch.zeros((1, E + (1 if shared else 0)), device=DEV)
    lg[0, E // 2] = float("inf")
    bad = layer.forward(x[:1].contiguous(), logits_in=lg)
    assert (bad["ids"] == -1).all() and torch.isnan(bad["y"]).all()
    assert bad["err"].cpu().numpy().tolist() == [1, 0, E // 2, 1, -1, 0]


# u in BF16 is the FP32 u rounded once: the same gates, products and sums on BF16-valued streams in either dtype (a gate
# a few 2^-24 off rounds some of these outputs the other way)
@pytest.mark.parametrize("bits,G,T,d,r", [(4, 64, 700, 2560, 320), (8, 64, 600, 1024, 128), (4, 32, 9, 2560, 96),
                                           (8, 64, 500, 2560, 128), (4, 64, 500, 2560, 512)])
def test_mix_up_bf16_is_the_rounded_fp32(bits, G, T, d, r):
    say("mix up bf16", bits, G, T, d, r)
    x = _bf16(orc.gen_bf16_normal(orc.tensor_key(12, "x"), 1.0, (T, 4 * d)))
    rng = np.random.default_rng(T)
    w = _weight(bits, 4 * d, r, G, 81)  # any codes: both calls read them chunk-major
    h, inv, nw = (torch.from_numpy(a.astype(np.float32)).to(DEV) for a in
                  (rng.standard_normal((T, r)), rng.uniform(0.5, 1.5, (T, 4)), rng.standard_normal(4 * d) * 0.1))
    assert torch.equal(moe.hc_mix_up(h, w, x, nw, inv), moe.hc_mix_up(h, w, x.float(), nw, inv).to(torch.bfloat16))


# a separate shared expert whose rows hold more groups than the GEMM's (H 4096, g 64), on either side of the sizes that
# go to the GEMM
@pytest.mark.parametrize("M", [100, 130])
def test_layer_shared_expert_of_many_groups(M):
    say("shared expert, H 4096", M)
    layer = moe.MoeLayer.synth(4096, 8, 2, 128, seed=5)
    x = moe.synth_bf16_normal(5, "x", 0, (M, 4096), 1.0)
    out = layer.forward(x)
    o = orc.moe_layer(oracle_weights(layer), to_np(x)[:16])
    assert np.array_equal(to_np(out["ids"])[:16], o["ids"])
    assert rel_err(to_np(out["y"])[:16], o["y"]) < 1e-2  # the layer tests' tolerance


# the up mix's variants: two blocks a CU and one, either format and dtype, ragged tokens, ranks on either side of the LDS
# that two blocks leave, group counts past the min terms held in registers
@pytest.mark.parametrize("bits,G,act,T,d,r", [(4, 64, "bf16", 497, 2560, 384), (4, 32, "f32", 497, 2560, 352),
                                              (8, 64, "bf16", 515, 2560, 128), (8, 32, "f32", 515, 2560, 96),
                                              (4, 64, "bf16", 431, 2560, 448), (8, 128, "bf16", 431, 2560, 768)])
def test_mix_up_kernels(bits, G, act, T, d, r):
    from oracle import hc

    say("mix up", bits, G, act, T, d, r)
    dt = torch.bfloat16 if act == "bf16" else torch.float32
    rng = np.random.default_rng(T)
    x = torch.from_numpy(rng.standard_normal((T, 4 * d)).astype(np.float32)).to(DEV).to(dt)
    h, inv, nw = (torch.from_numpy(a.astype(np.float32)).to(DEV) for a in
                  (rng.standard_normal((T, r)), rng.uniform(0.5, 1.5, (T, 4)), rng.standard_normal(4 * d) * 0.1))
    q, s, m = orc.gen_q(bits, orc.tensor_key(82, "gu_q"), orc.tensor_key(82, "gu_s"), 4 * d, r, G)
    w64 = hc.weights64(bits, q, s, m, 4 * d, r, G)
    u = moe.hc_mix_up(h, moe.QWeight.from_host(bits, *hc.to_chunk_major(bits, q, s, m, 4 * d, r, G), 4 * d, r, G), x, nw, inv)
    rows = np.unique(np.concatenate([np.arange(40), np.arange(T - 40, T)]))
    np64 = [t.double().cpu().numpy() for t in (h, x, nw, inv)]
    ref = hc.hc_mix_up(np64[0][rows], w64, np64[1][rows], np64[2], np64[3][rows], d)
    assert _rel64(u[rows], ref) < (2.0 ** -8 if act == "bf16" else 1e-4)  # one rounding of u; the gates' sums in FP32


# the per-slot combine: K whole, split over 4 and over 8 waves, slots within one round of waves and past it, a ragged
# column end; the grouped combine's bits, float64, the first invalid id of a token reported
# (and four waves a block, past two blocks a CU)
@pytest.mark.parametrize("G,K,A,N", [(128, 512, 17, 48), (128, 512, 5, 16), (128, 1024, 9, 32), (32, 1024, 3, 80),
                                     (128, 512, 6, 2816), (32, 1024, 3, 2816)])
def test_perslot_combine_rounds(G, K, A, N):
    say("per-slot combine", G, K, A, N)
    M, E = 3, 24
    w = _weight(4, E * N, K, G, 91)
    w64 = _w64(w)
    rng = np.random.default_rng(K + A)
    h = torch.from_numpy(rng.standard_normal((M * A, K)).astype(np.float32)).to(DEV)
    coef = torch.from_numpy(rng.random((M, A)).astype(np.float32)).to(DEV)
    ids = np.stack([rng.permutation(E)[:A] for _ in range(M)]).astype(np.int32)
    ids[1, A - 2], ids[1, A - 1] = E, -1
    tid = torch.from_numpy(ids).to(DEV)
    ws, _ = moe.moe_group_routes(tid, E)
    err = moe.zero_err()
    y = moe.experts_combine(h, w, E, tid, coef, err)
    yg = moe.experts_combine_grouped(h, w, E, tid, coef, ws, M, A)
    assert err.cpu().numpy().tolist() == [1, E, A + A - 2]
    assert torch.isnan(y[1]).all() and torch.equal(torch.nan_to_num(y, nan=7.0), torch.nan_to_num(yg, nan=7.0))
    h64, c64 = h.double().cpu().numpy(), coef.double().cpu().numpy()
    for m in (0, 2):
        ref = sum(c64[m, a] * (h64[m * A + a] @ w64[ids[m, a] * N:(ids[m, a] + 1) * N].T) for a in range(A))
        assert _rel64(y[m], ref) < 2e-5  # exact products, FP32 sums whose terms reach a few times the result


# the wave an output element of small calls and the tiles, on either side of the line between them: FP32 dense (K of one and
# several rounds of the lanes, a ragged last one, each format), and Q5 experts in BF16 grouped and per slot
@pytest.mark.parametrize("bits,G,K,N,M", [(4, 128, 128, 16, 1), (4, 64, 2112, 48, 9), (4, 64, 2112, 48, 90), (8, 64, 4160, 32, 3),
                                          (8, 32, 96, 64, 40), (8, 64, 512, 1024, 1), (8, 64, 512, 1024, 30)])
def test_small_fp32_dense(bits, G, K, N, M):
    say("small fp32 dense", bits, G, K, N, M)
    w = _weight(bits, N, K, G, 95)
    x = torch.from_numpy(np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)).to(DEV)
    ref = x.double().cpu().numpy() @ _w64(w).T
    lin = moe.linear_q4 if bits == 4 else moe.linear_q8
    y = lin(x, w, out_dtype=torch.float32)
    assert _rel64(y, ref) < 2e-5  # FP32 sums of up to 4160 terms
    assert torch.equal(lin(x, w, out_dtype=torch.bfloat16), y.to(torch.bfloat16))


@pytest.mark.parametrize("M,A", [(1, 3), (40, 3)])
def test_small_q5_bf16_experts(M, A):
    from oracle import q5

    say("small q5", M, A)
    E, H, I = 8, 2176, 64
    N = E * 2 * I
    q, s, m = q5.quantize((np.random.default_rng(1).standard_normal((N, H)) * 0.05).astype(np.float32), 128)
    gu, g64 = moe.QWeight.from_host(5, q, s, m, N, H, 128), q5.weights64(q, s, m, N, H, 128)
    x = _bf16(orc.gen_bf16_normal(orc.tensor_key(13, "x"), 1.0, (M, H)))
    ids = np.stack([np.random.default_rng(m).permutation(E)[:A] for m in range(M)]).astype(np.int32)
    tid = torch.from_numpy(ids).to(DEV)
    ws, _ = moe.moe_group_routes(tid, E)
    h = moe.experts_gather_grouped_swiglu(x, gu, E, ws, M, A)
    X = x.double().cpu().numpy()
    z = np.stack([X[s // A] @ g64[e * 2 * I:(e + 1) * 2 * I].T for s, e in enumerate(ids.ravel())])
    assert _rel64(h, z[:, :I] / (1 + np.exp(-z[:, :I])) * z[:, I:]) < 2.0 ** -8  # one BF16 rounding
    assert torch.equal(moe.experts_gather(x, gu, E, tid, moe.zero_err(), swiglu=True), h)


# the served widths (H 2560, I 640) with a separate shared expert - its split-K parts ride in the gate_up's and the down's
# launches - and the prefill router there, on either side of the logits from which it selects from the approximate pass; and
# the shared expert beside other counts of waves and groups
@pytest.mark.parametrize("H,I,M,E,k,shared", [
    (2560, 640, 1, 24, 6, True), (2560, 640, 11, 24, 6, True), (2560, 640, 16, 40, 10, True),
    (2560, 640, 300, 512, 10, "stacked"), (2560, 640, 257, 512, 4, False), (2560, 640, 300, 128, 10, True),
    (2304, 384, 7, 24, 6, True), (2816, 256, 16, 24, 4, True), (2304, 1024, 3, 24, 6, True), (2816, 896, 1, 24, 6, True)])
def test_layer_at_the_streamed_widths(H, I, M, E, k, shared):
    say("streamed widths", H, I, M, E, k, shared)
    layer = moe.MoeLayer.synth(H, E, k, I, seed=9, shared=shared)
    x = moe.synth_bf16_normal(9, "x", 0, (M, H), 1.0)
    out = layer.forward(x)
    rows = np.unique(np.concatenate([np.arange(min(M, 8)), np.arange(max(0, M - 8), M)]))
    o = orc.moe_layer(oracle_weights(layer), to_np(x)[rows])
    assert np.array_equal(to_np(out["ids"])[rows], o["ids"])
    assert rel_err(to_np(out["y"])[rows], o["y"]) < 1e-2  # the layer tests' tolerance


# nonzero-mean activations, and codes of a narrow part of their range. The tiles add codes 16 + n times x and take the offset out
# after: a group's running sum reaches 31 sum |x|, and is rounded at 2^-24 of that some eight times (four products of 32
# codes, the offset, the scale, the min, the accumulator), whatever the result's own size
@pytest.mark.parametrize("M,K,low", [(1, 3072, False), (64, 3072, False), (64, 3072, True), (1, 2048, True)])
def test_fp32_dense_off_centre(M, K, low):
    say("off centre", M, K, low)
    N, G = 512, 128
    rng = np.random.default_rng(M + K)
    codes = rng.integers(0, 3 if low else 16, size=(N, K)).astype(np.uint8)
    s = orc.f32_to_bf16(rng.uniform(0.01, 0.03, N * (K // G)).astype(np.float32))
    m = np.zeros_like(s) if low else orc.f32_to_bf16(orc.bf16_to_f32(s) * np.float32(-7.5))
    w = moe.QWeight.from_host(4, (codes[:, 0::2] | codes[:, 1::2] << 4).reshape(-1), s, m, N, K, G)
    x = (rng.standard_normal((M, K)) * 0.5 + 1).astype(np.float32)
    w64 = _w64(w)
    got = moe.linear_q4(torch.from_numpy(x).to(DEV), w, out_dtype=torch.float32).double().cpu().numpy()
    bound = 8 * 2.0 ** -24 * 31 * 0.03 * np.abs(x).sum(axis=1, keepdims=True)
    assert (np.abs(got - x.astype(np.float64) @ w64.T) < bound).all()
