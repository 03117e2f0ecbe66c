"""Prefill path on the GPU (BASELINE config 3 semantics) against the oracle: moe_align bit for bit, the grouped
gate/up/down within the bf16 rounding of h, the rank-order combine bit for bit, and the routed output within the
north-star bound against the fp64 exact-dequant reference."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from slotstream_spark_amd import _lib
from slotstream_spark_amd.engine.prefill import MoEPrefillLayer
from slotstream_spark_amd.kernels.fused_moe_affine import BLOCK_M, align_rows, combine_rank_order, fused_moe_affine
from slotstream_spark_amd.kernels.moe_align import moe_align
from slotstream_spark_amd.kernels.router import gemm_bf16
from slotstream_spark_amd.memory.synth import LayerWeights, normal_bf16, zipf_bias
from tests.gpu_util import DenseCache, bits, make_pool, rand_ids, rand_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,nl,bm,seed", [(0, 4, 64, 0), (1, 1, 64, 1), (37, 5, 4, 2), (1000, 32, 64, 3),
                                          (4099, 7, 16, 4), (20480, 512, 64, 5)])
def test_moe_align_matches_oracle(R, nl, bm, seed):
    print(f"[align] R={R} nl={nl} bm={bm}", flush=True)
    rng = np.random.default_rng(seed)
    le = rng.integers(-1, nl + 1, size=R).astype(np.int32)  # includes -1 and out-of-range entries
    if R > 10000:  # skewed, as Zipf routing makes it
        le = np.minimum(rng.zipf(1.3, size=R) - 1, nl - 1).astype(np.int32)
    s, b, n = moe_align(torch.from_numpy(le).cuda(), nl, bm)
    torch.cuda.synchronize()
    rs, rb, rn = O.moe_align(le, nl, bm)
    assert int(n.item()) == rn
    assert np.array_equal(s.cpu().numpy(), rs)
    assert np.array_equal(b.cpu().numpy(), rb)


@pytest.mark.parametrize("R,nl,bm", [(1024, 1024, 64), (1025, 1024, 64), (1024, 1025, 8), (5000, 4096, 16), (2049, 3, 128),
                                     (700, 1, 1), (1, 1024, 1024), (1000, 512, 128), (65536, 1024, 8), (66000, 1024, 8)])
def test_moe_align_one_and_three_launches(R, nl, bm):
    """Up to 1024 rows and experts the plan is one workgroup, past that three launches over 1024-row chunks; past 1024
    experts or 65,536 counts the offsets over the chunks are a launch of their own."""
    print(f"[align] R={R} nl={nl} bm={bm}", flush=True)
    rng = np.random.default_rng(R + nl)
    le = np.minimum(rng.zipf(1.2, size=R) - 2, nl).astype(np.int32)  # -1 and nl: skipped
    s, b, n = moe_align(torch.from_numpy(le).cuda(), nl, bm)
    torch.cuda.synchronize()
    rs, rb, rn = O.moe_align(le, nl, bm)
    assert int(n.item()) == rn
    assert np.array_equal(s.cpu().numpy(), rs)
    assert np.array_equal(b.cpu().numpy(), rb)


def _prefill_case(T, K, E, H, I, seed):
    pool = make_pool(E, H, I, seed=seed)
    x = normal_bf16((T, H), 1.0, seed + 1)
    ids = rand_ids(T, K, E, seed + 2).cuda()
    w = rand_weights(T, K, seed + 3).cuda()
    return pool, x, ids, w


def _oracle_rows(pool, x, ids, w, bf16_weights=True):
    H, I = pool.hidden, pool.inter
    cache = DenseCache(pool)
    dense = {}

    def weights_of(e):
        if e not in dense:
            rec = cache.record(e)
            dense[e] = O.expert_bf16(rec, H, I) if bf16_weights else O.expert_dense(rec, H, I, np.float64)
        return dense[e]
    T, K = ids.shape
    R = T * K
    return O.prefill_rows(O.bf16_to_f32(bits(x)), np.arange(R) // K, w.cpu().numpy().reshape(-1),
                          ids.cpu().numpy().reshape(-1), weights_of)


@pytest.mark.parametrize("T,K,E,H,I", [(50, 4, 16, 256, 128), (64, 10, 512, 2048, 512), (130, 10, 64, 2048, 512)])
def test_moe_prefill_matches_oracle(T, K, E, H, I):
    print(f"[prefill] T={T} K={K} E={E} H={H} I={I}", flush=True)
    pool, x, ids, w = _prefill_case(T, K, E, H, I, 1729 + T)
    lw = LayerWeights(H, E, 64, seed=7)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K, max_tokens=T)
    routed = layer.routed_experts(x, ids, w)
    torch.cuda.synchronize()
    assert _lib.device_error() == 0
    h_ref, rows_ref = _oracle_rows(pool, x, ids, w)
    R = T * K
    h = layer.h_buf[:R].float().cpu().numpy()
    rows = layer.out_rows[:R].cpu().numpy()
    same_h = float(np.mean(h == h_ref))
    err_rows = O.rel_l2(rows, rows_ref)
    print(f"h bf16 equal {same_h:.4f}; out_rows rel_l2 {err_rows:.2e}")
    assert same_h > 0.98            # h differs only where fp32 vs fp64 accumulation crosses a bf16 rounding edge
    assert err_rows < 2e-3
    # the combine is the sequential fp32 rank-order sum of the GPU's own rows, bit for bit
    assert np.array_equal(routed.cpu().numpy(), O.combine_rank_order(rows, T, K))
    # north star: within 2e-2 of the fp64 exact-dequant routed output
    _, rows64 = _oracle_rows(pool, x, ids, w, bf16_weights=False)
    err = O.rel_l2(routed.cpu().numpy(), O.combine_rank_order(rows64, T, K))
    print(f"routed vs exact-dequant fp64 rel_l2 {err:.2e}")
    assert err < 2e-2


def test_prefill_rows_independent_of_batch():
    """A row's output depends on that row and its record only (fused_moe_affine.py:1-20 contract)."""
    T, K, E, H, I = 96, 4, 8, 256, 128
    pool, x, ids, w = _prefill_case(T, K, E, H, I, 99)
    lw = LayerWeights(H, E, 64, seed=3)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K, max_tokens=T)
    layer.routed_experts(x, ids, w)
    full = layer.out_rows[:T * K].clone()
    half = T // 3
    layer.routed_experts(x[:half].contiguous(), ids[:half].contiguous(), w[:half].contiguous())
    torch.cuda.synchronize()
    assert torch.equal(layer.out_rows[:half * K], full[:half * K])


@pytest.mark.parametrize("H,I", [(256, 128), (512, 384), (2560, 640)])
def test_prefill_rows_same_bits_for_every_tile_shape(H, I):
    """Gate/up and down take two or four weight fragments per wave and one or two down tiles per block by the number of
    rows; live fragments and steps per LDS stage follow the rows of a block. A row's bits are the same under all of
    them (steps of 128 K: 2 to 20, odd at I 384 and 640), and agree with the oracle."""
    T, K, E = 2100, 4, 8
    pool, x, ids, w = _prefill_case(T, K, E, H, I, 7 * H + I)
    lw = LayerWeights(H, E, 64, seed=3)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K, max_tokens=T)
    layer.routed_experts(x, ids, w)                      # R = 8400: four fragments, two down tiles where H allows
    torch.cuda.synchronize()
    h_full, rows_full = layer.h_buf[:T * K].clone(), layer.out_rows[:T * K].clone()
    for t in (1, 3, 4, 20, 31, 33, 45, 64, 100, 150, 190, 230, 300):  # R 4 .. 1200: up to 150 rows per expert
        layer.h_buf.fill_(7.0)
        layer.out_rows.fill_(7.0)
        layer.routed_experts(x[:t].contiguous(), ids[:t].contiguous(), w[:t].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(layer.h_buf[:t * K], h_full[:t * K]), t
        assert torch.equal(layer.out_rows[:t * K], rows_full[:t * K]), t
        assert bool((layer.out_rows[t * K:] == 7.0).all()), t
    t = 60
    _, rows_ref = _oracle_rows(pool, x[:t].contiguous(), ids[:t].contiguous(), w[:t].contiguous())
    assert O.rel_l2(rows_full[:t * K].cpu().numpy(), rows_ref) < 2e-3


@pytest.mark.parametrize("I", [512, 768])
def test_down_rows_accumulate_in_the_dense_gemms_order(I):
    """The grouped GEMM adds up a row in the order of the dense GEMM (MFMA slices of 16 q + 8 s .. + 7 inside 64 K):
    with unit row weights its fp32 rows, rounded to bf16, are the dense product of the same h and the dequantized
    weights, bit for bit. Another order of the fp32 sums would flip some of the rounded values. Experts of 3 to 300 rows
    take every number of live fragments; I 768 has an odd number of 8-group chunks."""
    H, counts = 1024, [3, 20, 40, 60, 90, 128, 300]
    E, R = len(counts), sum(counts)
    print(f"[K order] I={I}", flush=True)
    pool = make_pool(E, H, I, seed=I)
    x = normal_bf16((R, H), 1.0, I + 1)
    row_expert = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32).cuda()
    gptr = pool.slot_ptr[pool.map[:E].long()].contiguous()
    h = torch.empty((R, I), dtype=torch.bfloat16, device="cuda")
    out_rows = torch.empty((R, H), device="cuda")
    fused_moe_affine(x, torch.arange(R, dtype=torch.int32, device="cuda"), torch.ones(R, device="cuda"),
                     torch.arange(E, dtype=torch.int32, device="cuda"), gptr, out_rows, row_expert=row_expert, h_buf=h)
    cache, r0 = DenseCache(pool), 0
    for e, n in enumerate(counts):
        down = torch.from_numpy(O.expert_bf16(cache.record(e), H, I)[2]).to(torch.bfloat16).cuda()
        ref = gemm_bf16(h[r0:r0 + n].contiguous(), down)
        assert torch.equal(out_rows[r0:r0 + n].to(torch.bfloat16), ref), (e, n)
        r0 += n


def test_fused_moe_affine_group_semantics():
    """The reference interface: a group of local experts through expert_map; rows outside it are left alone."""
    T, K, E, H, I = 40, 4, 12, 256, 128
    pool, x, ids, w = _prefill_case(T, K, E, H, I, 5)
    group = [1, 4, 7, 9]
    emap = torch.full((E,), -1, dtype=torch.int32)
    emap[group] = torch.arange(len(group), dtype=torch.int32)
    slots = pool.map.cpu()
    gptr = torch.tensor([int(pool.slot_ptr[int(slots[e])]) for e in group], dtype=torch.int64).cuda()
    R = T * K
    row_expert = ids.reshape(-1).contiguous()
    row_token = (torch.arange(R, device="cuda") // K).to(torch.int32)
    row_weight = w.reshape(-1).contiguous()
    out_rows = torch.full((R, H), 7.0, device="cuda")
    fused_moe_affine(x, row_token, row_weight, emap.cuda(), gptr, out_rows, row_expert=row_expert, inter=I)
    torch.cuda.synchronize()
    _, rows_ref = _oracle_rows(pool, x, ids, w)
    in_group = np.isin(row_expert.cpu().numpy(), group)
    got = out_rows.cpu().numpy()
    assert np.all(got[~in_group] == 7.0)
    assert O.rel_l2(got[in_group], rows_ref[in_group]) < 2e-3
    s, b, n = align_rows(row_expert, emap.cuda(), len(group))
    rs, rb, rn = O.moe_align(np.where(in_group, emap.numpy()[row_expert.cpu().numpy()], -1), len(group), BLOCK_M)
    assert np.array_equal(s.cpu().numpy(), rs) and int(n.item()) == rn


@pytest.mark.parametrize("counts,blocks", [
    ([0, 0, 1, 0, 0, 0, 0, 1, 0, 1, 1, 1], None),          # one block per expert, empty ones included
    # blocks without rows, then an expert's rows one to a block
    ([12] + [0] * 19, [(e, 0, 0) for e in range(8)] + [(0, r, 1) for r in range(12)]),
    ([0, 130, 2], [(0, 0, 0), (1, 0, 128), (1, 128, 2), (2, 130, 2)]),
])
def test_fused_moe_affine_takes_plans_with_more_blocks(counts, blocks):
    """A caller's plan may have as many blocks as padded_rows holds, more than the rows need: all of them are computed,
    with the bits of the aligned plan."""
    E, R, H, I = len(counts), sum(counts), 256, 128
    print(f"[plan] counts={counts}", flush=True)
    if blocks is None:
        starts = np.concatenate([[0], np.cumsum(counts)])
        blocks = [(e, int(starts[e]), counts[e]) for e in range(E)]
    P = int(_lib.lib().ssmoe_padded_rows(R, E, BLOCK_M))
    assert len(blocks) * BLOCK_M <= P
    sorted_rows, block_expert = np.full(P, R, np.int32), np.full(P // BLOCK_M, -1, np.int32)
    for b, (e, r0, n) in enumerate(blocks):
        block_expert[b] = e
        sorted_rows[b * BLOCK_M: b * BLOCK_M + n] = np.arange(r0, r0 + n)
    plan = tuple(torch.from_numpy(t).cuda() for t in (sorted_rows, block_expert,
                                                      np.array([len(blocks) * BLOCK_M], np.int32)))
    pool = make_pool(E, H, I, seed=E)
    x = normal_bf16((R, H), 1.0, E + 1)
    row_expert = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32).cuda()
    emap, gptr = torch.arange(E, dtype=torch.int32, device="cuda"), pool.slot_ptr[pool.map[:E].long()].contiguous()
    got = []
    for aligned in (None, plan):
        h = torch.full((R, I), 7.0, dtype=torch.bfloat16, device="cuda")
        out_rows = torch.full((R, H), 7.0, device="cuda")
        fused_moe_affine(x, torch.arange(R, dtype=torch.int32, device="cuda"), torch.ones(R, device="cuda"), emap, gptr,
                         out_rows, row_expert=row_expert, h_buf=h, aligned=aligned)
        got.append((h, out_rows))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def test_combine_rank_order_bitwise():
    T, K, H = 33, 10, 2048
    g = torch.Generator(device="cuda").manual_seed(1)
    rows = torch.randn((T * K, H), generator=g, device="cuda") * 3
    out = combine_rank_order(rows, T, K)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), O.combine_rank_order(rows.cpu().numpy(), T, K))


@pytest.mark.parametrize("T", [9, 700])
def test_prefill_skipped_rows_in_both_plans(T):
    """Ids out of range and experts that are not resident are skipped (+0 in the sum) and flagged, in the one-workgroup
    plan and in the chunked one."""
    K, E, H, I = 2, 8, 256, 128
    pool, x, ids, w = _prefill_case(T, K, E, H, I, 13)
    pool.map[5] = -1
    lw = LayerWeights(H, E, 64, seed=2)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K, max_tokens=T)
    ids = ids.clone()
    ids[2, 1], ids[T - 1, 0] = -3, E
    _lib.device_error()
    routed = layer.routed_experts(x, ids, w)
    torch.cuda.synchronize()
    assert _lib.device_error() & 3 == 3
    flat = ids.cpu().numpy().reshape(-1)
    ok = (flat >= 0) & (flat < E) & (flat != 5)
    _, rows_ref = _oracle_rows(pool, x, torch.from_numpy(np.where(ok, flat, -1).reshape(T, K)), w)
    assert O.rel_l2(routed.cpu().numpy(), O.combine_rank_order(rows_ref, T, K)) < 2e-3


def test_prefill_unmapped_expert_flagged():
    T, K, E, H, I = 8, 2, 8, 256, 128
    pool, x, ids, w = _prefill_case(T, K, E, H, I, 11)
    lw = LayerWeights(H, E, 64, seed=2)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K, max_tokens=T)
    ids = ids.clone()
    ids[3, 1] = E + 5
    _lib.device_error()
    routed = layer.routed_experts(x, ids, w)
    torch.cuda.synchronize()
    assert _lib.device_error() & 1
    ids_c = ids.cpu().numpy().reshape(-1)
    _, rows_ref = _oracle_rows(pool, x, torch.from_numpy(np.where(ids_c < E, ids_c, -1).reshape(T, K)), w)
    ref = O.combine_rank_order(rows_ref, T, K)
    assert O.rel_l2(routed.cpu().numpy(), ref) < 2e-3


def test_prefill_layer_end_to_end():
    """Router (bf16 MFMA GEMM + device top-k) + routed experts + shared expert at the config-3 shape on a short chunk;
    the GEMMs themselves are checked in test_gpu_dense_gemm.py."""
    T, K, E, H, I = 128, 10, 512, 2048, 512
    pool = make_pool(E, H, I, seed=31)
    lw = LayerWeights(H, E, 512, seed=32)
    bias = zipf_bias(E, 1.1, 1731)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K,
                            router_bias=bias, max_tokens=T)
    x = normal_bf16((T, H), 1.0, 33)
    y, ids, w, routed = layer(x)
    torch.cuda.synchronize()
    # routing against the oracle's router tail applied to the GEMM's own logits
    logits = gemm_bf16(x, lw.router_w)
    _, rids, rw = O.router_topk(bits(logits), K, bias.cpu().numpy())
    assert np.array_equal(ids.cpu().numpy(), rids)
    assert np.array_equal(w.cpu().numpy().view(np.uint32), rw.view(np.uint32))
    _, rows_ref = _oracle_rows(pool, x, ids, w)
    assert O.rel_l2(routed.cpu().numpy(), O.combine_rank_order(rows_ref, T, K)) < 2e-3
    # the shared expert's elementwise chain and y, bit for bit, from the GEMMs' own bf16 outputs
    proj = gemm_bf16(x, layer.sh_cat)
    Is = lw.sh_gate.shape[0]
    pb = bits(proj)
    hs_ref = O.shared_hs(pb[:, :Is], pb[:, Is:2 * Is])
    sh = gemm_bf16(torch.from_numpy(hs_ref.view(np.int16)).view(torch.bfloat16).cuda(), lw.sh_down)
    y_ref = O.combine_shared(routed.cpu().numpy(), bits(sh), pb[:, 2 * Is].copy())
    assert np.array_equal(bits(y), y_ref)
    assert torch.isfinite(y.float()).all()


@pytest.mark.parametrize("T,E,H,Is", [(1, 8, 256, 256), (33, 64, 512, 256), (70, 520, 2048, 512), (300, 64, 256, 768),
                                      (1100, 512, 512, 512), (2049, 512, 256, 512), (1800, 520, 512, 512)])
def test_prefill_layer_equals_its_parts(T, E, H, Is):
    """The layer in one C call against the separate calls, bit for bit. Its input projections take the 32 x 64 tile in the
    first three cases, 64 x 64 in the next two and 128 x 128 in the last two (17 x 13 and 15 x 13 tiles); T and the
    router's columns are ragged."""
    K, I = 4, 128
    pool = make_pool(E, H, I, seed=T)
    lw = LayerWeights(H, E, Is, seed=T + 1)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K,
                            router_bias=zipf_bias(E, 1.1, 3), max_tokens=T)
    x = normal_bf16((T, H), 1.0, T + 2)
    ids, w = (t.clone() for t in layer.route(x))
    routed = layer.routed_experts(x, ids, w).clone()
    sh, sgl = layer.shared(x)
    y = torch.empty((T, H), dtype=torch.bfloat16, device="cuda")
    _lib.check(_lib.lib().ssmoe_combine_shared(routed.data_ptr(), sh.data_ptr(), sgl.data_ptr(), y.data_ptr(), T, H,
                                               torch.cuda.current_stream().cuda_stream))
    got = layer(x)
    torch.cuda.synchronize()
    for g, ref in zip(got, (y, ids, w, routed)):
        assert torch.equal(g, ref)


@pytest.mark.parametrize("T,Is,ld", [(1, 8, 17), (37, 512, 1032), (300, 640, 1288)])
def test_shared_hs_bitwise(T, Is, ld):
    g = torch.Generator(device="cuda").manual_seed(T)
    proj = (torch.randn((T, ld), generator=g, device="cuda") * 4).to(torch.bfloat16)
    hs = torch.empty((T, Is), dtype=torch.bfloat16, device="cuda")
    sgl = torch.empty((T,), dtype=torch.bfloat16, device="cuda")
    _lib.check(_lib.lib().ssmoe_shared_hs(proj.data_ptr(), ld, T, Is, hs.data_ptr(), sgl.data_ptr(), 0))
    torch.cuda.synchronize()
    pb = bits(proj)
    assert np.array_equal(bits(hs), O.shared_hs(pb[:, :Is], pb[:, Is:2 * Is]))
    assert np.array_equal(bits(sgl), pb[:, 2 * Is])


@pytest.mark.parametrize("T,H", [(1, 4), (33, 2048), (129, 2560)])
def test_combine_shared_bitwise(T, H):
    g = torch.Generator(device="cuda").manual_seed(H + T)
    routed = torch.randn((T, H), generator=g, device="cuda") * 3
    sh = (torch.randn((T, H), generator=g, device="cuda")).to(torch.bfloat16)
    sgl = (torch.randn((T,), generator=g, device="cuda") * 5).to(torch.bfloat16)
    y = torch.empty((T, H), dtype=torch.bfloat16, device="cuda")
    _lib.check(_lib.lib().ssmoe_combine_shared(routed.data_ptr(), sh.data_ptr(), sgl.data_ptr(), y.data_ptr(), T, H, 0))
    torch.cuda.synchronize()
    assert np.array_equal(bits(y), O.combine_shared(routed.cpu().numpy(), bits(sh), bits(sgl)))


def test_moe_prefill_config3_full_size():
    """BASELINE config 3 at its own size: 2048 tokens through the config-1 layer (E=512, top-10), routed by the
    oracle's router with the Zipf(1.1) bias, so the head experts hold many 128-row M blocks each (reached through
    block_expert and the XCD-contiguous tile order) and the tail experts a few rows. Every routed row against the
    oracle (fused_moe_affine.py:136-172, moe_sweep.py:80-176 semantics), the combine bit for bit, the routed output
    within the north-star bound of the fp64 exact-dequant reference."""
    T, K, E, H, I = 2048, 10, 512, 2048, 512
    print(f"[prefill config3] T={T} K={K} E={E}", flush=True)
    pool = make_pool(E, H, I, seed=2048)
    lw = LayerWeights(H, E, 512, seed=2049)
    bias = zipf_bias(E, 1.1, 1731)
    x = normal_bf16((T, H), 1.0, 2050)
    _, _, rids, rwt = O.router(bits(x), bits(lw.router_w), K, bias.cpu().numpy())
    counts = np.bincount(rids.reshape(-1), minlength=E)
    print(f"experts touched {int((counts > 0).sum())}, rows of the largest {int(counts.max())}", flush=True)
    assert counts.max() >= 4 * BLOCK_M                       # an expert spanning at least four M blocks
    assert ((counts > 0) & (counts < BLOCK_M)).sum() >= 10   # and many single-block experts
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K,
                            router_bias=bias, max_tokens=T)
    ids, w = torch.from_numpy(rids).cuda(), torch.from_numpy(rwt).cuda()
    routed = layer.routed_experts(x, ids, w)
    torch.cuda.synchronize()
    assert _lib.device_error() == 0
    cache = DenseCache(pool)
    R = T * K
    xf = O.bf16_to_f32(bits(x))
    h_ref, rows_ref = O.prefill_rows(xf, np.arange(R) // K, rwt.reshape(-1), rids.reshape(-1),
                                     lambda e: O.expert_bf16(cache.record(e), H, I))
    h = layer.h_buf[:R].float().cpu().numpy()
    rows = layer.out_rows[:R].cpu().numpy()
    same_h = float(np.mean(h == h_ref))
    err_rows = O.rel_l2(rows, rows_ref)
    worst = max(O.rel_l2(rows[rids.reshape(-1) == e], rows_ref[rids.reshape(-1) == e]) for e in np.nonzero(counts)[0])
    print(f"h bf16 equal {same_h:.4f}; out_rows rel_l2 {err_rows:.2e}, worst expert {worst:.2e}", flush=True)
    assert same_h > 0.98
    assert err_rows < 2e-3 and worst < 4e-3
    assert np.array_equal(routed.cpu().numpy(), O.combine_rank_order(rows, T, K))
    del h_ref, rows_ref
    _, rows64 = O.prefill_rows(xf, np.arange(R) // K, rwt.reshape(-1), rids.reshape(-1),
                               lambda e: O.expert_dense(cache.record(e), H, I, np.float64))
    err = O.rel_l2(routed.cpu().numpy(), O.combine_rank_order(rows64, T, K))
    print(f"routed vs exact-dequant fp64 rel_l2 {err:.2e}")
    assert err < 2e-2


@pytest.mark.parametrize("T,H", [(6900, 2560), (8193, 2048)])
def test_prefill_streamed_rows_equal_plain_rows(T, H):
    """Past 256 MB of out_rows the down product stores them non-temporally. Rows and sums are bit for bit those of the
    same tokens in chunks below that (T K H 4 = 283 MB and 268 MB + 32 KB, chunks of 40 MB and less)."""
    K, E, I = 4, 8, 128
    print(f"[streamed rows] T={T} H={H}", flush=True)
    pool, x, ids, w = _prefill_case(T, K, E, H, I, 11 * H + T)
    lw = LayerWeights(H, E, 64, seed=3)
    layer = MoEPrefillLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=K, max_tokens=T)
    assert T * K * H * 4 > 256 << 20
    full = layer.routed_experts(x, ids, w).clone()
    rows = layer.out_rows[:T * K].clone()
    for t0 in range(0, T, 1000):
        t1 = min(T, t0 + 1000)
        layer.out_rows.fill_(7.0)
        part = layer.routed_experts(x[t0:t1].contiguous(), ids[t0:t1].contiguous(), w[t0:t1].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(layer.out_rows[:(t1 - t0) * K], rows[t0 * K:t1 * K]), t0
        assert torch.equal(part, full[t0:t1]), t0
