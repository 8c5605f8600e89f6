"""GPU parity of the fused encode kernel (bit-exact).

Pins: the committed torch fixtures (tests/golden/encode_golden.npz, torch CPU
running spherical_kv_pipeline.py:1136-1144 + pagebuilder.py:8-33) and the C
oracle on the full config-3 workload.
"""
import os

import numpy as np
import pytest
import torch

import oracle
import sphkv_format as fmt
import sphkv_ops as ops
import sphkv_synth as synth
from gpu_helpers import log, single_page_plan

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def test_encode_golden_fixtures(gpu):
    z = np.load(os.path.join(GOLD, "encode_golden.npz"))
    names = sorted({k.split("__")[0] for k in z.files if "__" in k})
    for name in names:
        N, tid, g, b, dh = (int(x) for x in z[name + "__meta"])
        log(f"encode fixture {name} N={N} tier={tid} dh={dh}")
        plan = single_page_plan(N, tid, dh)
        pool = ops.PagedPool.allocate(plan, {tid: z[name + "__cb"][None]}, gpu)
        K = torch.as_tensor(z[name + "__K"], device=gpu)
        V = torch.zeros_like(K)
        src = torch.as_tensor(np.where(plan.tokens >= 0, plan.tokens, -1), device=gpu)
        r_out = torch.zeros((1, 16, dh // 16), dtype=torch.float32, device=gpu)
        c_out = torch.zeros((1, 16, dh // 16), dtype=torch.int32, device=gpu)
        ops.encode_pages(pool, K, V, src, r_out, c_out)
        torch.cuda.synchronize()
        G = dh // g
        page = pool.pages.cpu().numpy()[: z[name + "__page"].size]
        r = r_out.cpu().numpy()[0, :N, :G]
        c = c_out.cpu().numpy()[0, :N, :G]
        assert (r.view(np.uint32) == z[name + "__r"].view(np.uint32)).all(), name
        assert (c == z[name + "__codes"]).all(), name
        assert (page == z[name + "__page"]).all(), name


def test_encode_fp32_input_matches_fp16(gpu):
    # the reference feeds K.float(); fp32 input of the same values is identical
    z = np.load(os.path.join(GOLD, "encode_golden.npz"))
    name = "t1_n16_c3"
    plan = single_page_plan(16, 1, 128)
    outs = []
    for dt in (torch.float16, torch.float32):
        pool = ops.PagedPool.allocate(plan, {1: z[name + "__cb"][None]}, gpu)
        K = torch.as_tensor(z[name + "__K"], device=gpu).to(dt)
        ops.encode_pages(pool, K, torch.zeros(K.shape, dtype=torch.float16, device=gpu),
                         torch.as_tensor(plan.tokens, device=gpu))
        outs.append(pool.pages.cpu().numpy())
    assert (outs[0] == outs[1]).all()
    assert (outs[0][: z[name + "__page"].size] == z[name + "__page"]).all()


@pytest.mark.parametrize("config", [3, 2, 1])
def test_encode_full_workload_vs_oracle(gpu, config):
    wl = synth.make_encode_workload() if config == 3 else synth.make_decode_workload(config)
    log(f"encode full config{config}: rows={wl.plan.num_rows}")
    pool, r_out, c_out = ops.build_pool_gpu(wl, gpu, with_codes=True)
    torch.cuda.synchronize()
    cpu = oracle.build_pool(wl, with_codes=True)
    pages = pool.pages.cpu().numpy()
    assert (pages == cpu["pages"]).all(), f"{int((pages != cpu['pages']).sum())} page bytes differ"
    assert (pool.v_pool.cpu().numpy().view(np.uint16) == cpu["v_pool"].view(np.uint16)).all()
    r, c = r_out.cpu().numpy(), c_out.cpu().numpy()
    comp = wl.plan.tier != fmt.DENSE_TIER_ID
    assert (c[comp] == cpu["codes"][comp]).all()
    assert (r[comp].view(np.uint32) == cpu["r"][comp].view(np.uint32)).all()


def test_encode_partial_and_edge_pages(gpu):
    # ragged tier lists: pages with 1..16 tokens, tier 3, dense, dh 64 and 128
    rng = np.random.default_rng(11)
    for dh in (64, 128):
        L = 173
        tier_of = [rng.choice(np.array([1, 2, 3, fmt.DENSE_TIER_ID], np.int32), size=L) for _ in range(3)]
        cbs = synth.make_codebooks(rng, 3, dh, [1, 2, 3])
        K = [(rng.standard_normal((3, L, dh)) * 3).astype(np.float16)]
        V = [rng.standard_normal((3, L, dh)).astype(np.float16)]
        plan = fmt.plan_pages(tier_of, None, 1, 3, dh, 16, rng=rng, num_vpages=None)
        wl = synth.Workload(name="edge", dh=dh, num_kv=3, gqa=1, num_seqs=1, lengths=[L], rope_theta=5e5,
                            codebooks=cbs, K=K, V=V, q=np.zeros((1, 3, dh), np.float16), tier_of=tier_of,
                            plan=plan)
        log(f"encode edge dh={dh} rows={plan.num_rows} counts={sorted(set(plan.count.tolist()))}")
        pool, r_out, c_out = ops.build_pool_gpu(wl, gpu, with_codes=True)
        torch.cuda.synchronize()
        cpu = oracle.build_pool(wl, with_codes=True)
        assert (pool.pages.cpu().numpy() == cpu["pages"]).all()
        assert (pool.v_pool.cpu().numpy().view(np.uint16) == cpu["v_pool"].view(np.uint16)).all()


def test_encode_near_ties_and_degenerate_groups(gpu):
    # Keys built to stress the nearest-centroid search: the sum of two
    # centroids of the group (an exact tie in real arithmetic, decided by the
    # rounding of the reference's fp32 dot products), a centroid itself at
    # several scales, a centroid plus a tiny share of another, and all-zero
    # groups.  Codes and radii must match the C oracle bit for bit.
    rng = np.random.default_rng(23)
    dh, H, L = 128, 2, 160
    tier_of = [np.array([[1, 2, 3][(i + h) % 3] for i in range(L)], np.int32) for h in range(H)]
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    K = np.zeros((H, L, dh), np.float32)
    for h in range(H):
        for t in range(L):
            tid = int(tier_of[h][t])
            cb = cbs[tid][h]                      # [G, C, g]
            G, C, g = cb.shape
            for j in range(G):
                a, b = rng.choice(C, size=2, replace=False)
                kind = (t + j) % 5
                if kind == 0:
                    v = cb[j, a] + cb[j, b]
                elif kind == 1:
                    v = cb[j, a] * np.float32(2.0 ** rng.integers(-6, 7))
                elif kind == 2:
                    v = cb[j, a] + np.float32(1e-3) * cb[j, b]
                elif kind == 3:
                    v = np.zeros(g, np.float32)
                else:
                    v = (cb[j, a] - cb[j, b]) * np.float32(0.5)
                K[h, t, j * g:(j + 1) * g] = v
    K16 = [K.astype(np.float16)]
    V = [rng.standard_normal((H, L, dh)).astype(np.float16)]
    plan = fmt.plan_pages(tier_of, None, 1, H, dh, 16, rng=rng, num_vpages=None)
    wl = synth.Workload(name="ties", dh=dh, num_kv=H, gqa=1, num_seqs=1, lengths=[L], rope_theta=5e5,
                        codebooks=cbs, K=K16, V=V, q=np.zeros((1, H, dh), np.float16), tier_of=tier_of,
                        plan=plan)
    log(f"encode near-ties dh={dh} rows={plan.num_rows}")
    pool, r_out, c_out = ops.build_pool_gpu(wl, gpu, with_codes=True)
    torch.cuda.synchronize()
    cpu = oracle.build_pool(wl, with_codes=True)
    r, c = r_out.cpu().numpy(), c_out.cpu().numpy()
    comp = wl.plan.tier != fmt.DENSE_TIER_ID
    assert (c[comp] == cpu["codes"][comp]).all(), f"{int((c[comp] != cpu['codes'][comp]).sum())} codes differ"
    assert (r[comp].view(np.uint32) == cpu["r"][comp].view(np.uint32)).all()
    assert (pool.pages.cpu().numpy() == cpu["pages"]).all()


@pytest.mark.parametrize("kind", ["scaled", "raw", "near_unit"])
def test_encode_non_unit_codebooks_bit_exact(gpu, kind):
    # _encode_keys_with_codebooks (spherical_kv_pipeline.py:1130-1144) takes
    # any codebook; only codebook_loader.py:43-44 normalises the rows.  Rows
    # scaled by 0.5..3, raw N(0,1) rows, and rows 1% off unit length (inside
    # the pre-ranking bound) must all give the oracle's codes, radii and pages.
    rng = np.random.default_rng({"scaled": 31, "raw": 32, "near_unit": 33}[kind])
    dh, H, L = 128, 2, 200
    tier_of = [rng.choice(np.array([1, 2, 3], np.int32), size=L) for _ in range(H)]
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    for tid, cb in cbs.items():
        if kind == "scaled":
            cb *= rng.uniform(0.5, 3.0, size=cb.shape[:-1] + (1,)).astype(np.float32)
        elif kind == "raw":
            cb[:] = rng.standard_normal(cb.shape).astype(np.float32)
        else:
            cb *= np.float32(1.01)
    # keys on near-ties of the scaled rows: c_a + c_b and c_a + 1e-3 c_b, plus plain ones
    K = np.zeros((H, L, dh), np.float32)
    for h in range(H):
        for t in range(L):
            cb = cbs[int(tier_of[h][t])][h]
            G, C, g = cb.shape
            for j in range(G):
                a, b = rng.choice(C, size=2, replace=False)
                m = (t + j) % 3
                v = cb[j, a] + cb[j, b] if m == 0 else (cb[j, a] + np.float32(1e-3) * cb[j, b] if m == 1
                                                         else rng.standard_normal(g).astype(np.float32))
                K[h, t, j * g:(j + 1) * g] = v
    V = [rng.standard_normal((H, L, dh)).astype(np.float16)]
    plan = fmt.plan_pages(tier_of, None, 1, H, dh, 16, rng=rng, num_vpages=None)
    wl = synth.Workload(name=f"nonunit_{kind}", dh=dh, num_kv=H, gqa=1, num_seqs=1, lengths=[L], rope_theta=5e5,
                        codebooks=cbs, K=[K.astype(np.float16)], V=V, q=np.zeros((1, H, dh), np.float16),
                        tier_of=tier_of, plan=plan)
    log(f"encode non-unit codebooks ({kind}) rows={plan.num_rows}")
    pool, r_out, c_out = ops.build_pool_gpu(wl, gpu, with_codes=True)
    torch.cuda.synchronize()
    cpu = oracle.build_pool(wl, with_codes=True)
    r, c = r_out.cpu().numpy(), c_out.cpu().numpy()
    comp = wl.plan.tier != fmt.DENSE_TIER_ID
    assert (c[comp] == cpu["codes"][comp]).all(), f"{int((c[comp] != cpu['codes'][comp]).sum())} codes differ"
    assert (r[comp].view(np.uint32) == cpu["r"][comp].view(np.uint32)).all()
    assert (pool.pages.cpu().numpy() == cpu["pages"]).all()


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("dh,H,L", [(128, 2, 203), (64, 3, 77)])
def test_encode_small_gaps_scales_and_bit_patterns(gpu, dh, H, L, fp32):
    # the MFMA ranking and its exact pass: gaps of 1e-7 to 1e-2 between the two
    # best centroids (around the slack past which the ranking stands), ties of
    # three centroids, groups from zero and fp16 denormals to large, pages of every
    # tier mixed in one workgroup, missing rows at the end of a workgroup; V and
    # dense K of any bit pattern (negative zeros, infinities, NaNs) as they are
    rng = np.random.default_rng(dh + fp32)
    tier_of = [rng.choice(np.array([1, 2, 3, fmt.DENSE_TIER_ID], np.int32), size=L) for _ in range(H)]
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    K = np.zeros((H, L, dh), np.float32)
    for h in range(H):
        for t in range(L):
            tid = int(tier_of[h][t])
            if tid == fmt.DENSE_TIER_ID:
                K[h, t] = rng.integers(0, 1 << 16, dh).astype(np.uint16).view(np.float16).astype(np.float32)
                continue
            cb = cbs[tid][h]
            G, C, g = cb.shape
            for j in range(G):
                a, b, c = rng.choice(C, size=3, replace=False)
                eps = np.float32(10.0 ** rng.uniform(-7, -2))
                v = cb[j, a] + cb[j, b] * (1 - eps) + (cb[j, c] * (1 - eps) if t % 3 == 0 else 0)
                scale = np.float32(2.0 ** rng.integers(-22, 9)) if (t + j) % 13 else np.float32(0)   # 0 (and -0): a zero key
                K[h, t, j * g:(j + 1) * g] = v * scale
    dense = np.stack([t == fmt.DENSE_TIER_ID for t in tier_of])
    if fp32:
        K[dense] = np.where(np.isnan(K[dense]), 1.0, K[dense])       # (a NaN's payload is not kept by the conversion)
    V = rng.integers(0, 1 << 16, (H, L, dh)).astype(np.uint16).view(np.float16)
    plan = fmt.plan_pages(tier_of, None, 1, H, dh, 16, rng=rng)
    wl = synth.Workload(name="gaps", dh=dh, num_kv=H, gqa=1, num_seqs=1, lengths=[L], rope_theta=5e5, codebooks=cbs,
                        K=[K if fp32 else K.astype(np.float16)], V=[V], q=np.zeros((1, H, dh), np.float16),
                        tier_of=tier_of, plan=plan)
    log(f"encode gaps dh={dh} fp32={fp32} rows={plan.num_rows}")
    pool, r_out, c_out = ops.build_pool_gpu(wl, gpu, with_codes=True)
    torch.cuda.synchronize()
    cpu = oracle.build_pool(wl, with_codes=True)
    r, c = r_out.cpu().numpy(), c_out.cpu().numpy()
    comp = plan.tier != fmt.DENSE_TIER_ID
    assert (c[comp] == cpu["codes"][comp]).all(), f"{int((c[comp] != cpu['codes'][comp]).sum())} codes differ"
    assert (r[comp].view(np.uint32) == cpu["r"][comp].view(np.uint32)).all()
    assert (pool.pages.cpu().numpy() == cpu["pages"]).all()
    assert (pool.v_pool.cpu().numpy().view(np.uint16) == cpu["v_pool"].view(np.uint16)).all()


def _codes_and_radii(gpu, rng, K, tier_of, cbs, H, L, dh):
    plan = fmt.plan_pages(tier_of, None, 1, H, dh, 16, rng=rng)
    wl = synth.Workload(name="codes", dh=dh, num_kv=H, gqa=1, num_seqs=1, lengths=[L], rope_theta=5e5, codebooks=cbs,
                        K=[K], V=[np.zeros((H, L, dh), np.float16)], q=np.zeros((1, H, dh), np.float16),
                        tier_of=tier_of, plan=plan)
    pool, r_out, c_out = ops.build_pool_gpu(wl, gpu, with_codes=True)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        cpu = oracle.build_pool(wl, with_codes=True)
    return r_out.cpu().numpy(), c_out.cpu().numpy(), cpu


@pytest.mark.parametrize("fp32", [False, True])
def test_encode_infinite_keys_take_the_first_code(gpu, fp32):
    # a group with infinities has NaN directions and NaN similarities: the
    # first code wins, however the unnormalised products rank (several
    # infinities leave some of them -inf and the rest NaN)
    rng = np.random.default_rng(5)
    H, L, dh = 2, 400, 128
    tier_of = [rng.choice(np.array([1, 2, 3], np.int32), size=L) for _ in range(H)]
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    K = rng.standard_normal((H, L, dh)).astype(np.float32 if fp32 else np.float16)
    for h in range(H):
        for t in range(L):
            for j in range(0, dh, 16):
                n = int(rng.integers(0, 7))
                K[h, t, j + rng.choice(16, n, replace=False)] = np.inf * rng.choice([-1, 1], n)
    log(f"infinite keys fp32={fp32}")
    _, c, cpu = _codes_and_radii(gpu, rng, K, tier_of, cbs, H, L, dh)
    assert (c == cpu["codes"]).all(), f"{int((c != cpu['codes']).sum())} codes differ"


def test_encode_tiny_fp32_keys(gpu):
    # norms from where their squares are denormal (so that the fp32 norm is off
    # by up to a factor) to ordinary ones, gaps between the two best centroids
    # of 1e-6 to 1e-3
    rng = np.random.default_rng(6)
    H, L, dh = 2, 1500, 128
    tier_of = [rng.choice(np.array([1, 2, 3], np.int32), size=L) for _ in range(H)]
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    K = np.zeros((H, L, dh), np.float32)
    for h in range(H):
        for t in range(L):
            cb = cbs[int(tier_of[h][t])][h]
            G, C, g = cb.shape
            for j in range(G):
                a, b = rng.choice(C, size=2, replace=False)
                v = cb[j, a] + cb[j, b] * np.float32(1 - 10.0 ** rng.uniform(-6, -3))
                K[h, t, j * g:(j + 1) * g] = v * np.float32(10.0 ** rng.uniform(-23.2, -17 if t % 2 else -22))
    log("tiny fp32 keys")
    r, c, cpu = _codes_and_radii(gpu, rng, K, tier_of, cbs, H, L, dh)
    assert (r.view(np.uint32) == cpu["r"].view(np.uint32)).all()
    assert (c == cpu["codes"]).all(), f"{int((c != cpu['codes']).sum())} codes differ"


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("kind", ["one", "twice", "four", "last_value", "zero_sign"])
def test_encode_repeated_codebook_rows(gpu, kind, fp32):
    # ties of whole rows go to the first code; rows that differ in their last
    # value or in a zero's sign are scored like any others; pages of 1 token
    # (torch's M = 1 order) to 16, of every tier
    rng = np.random.default_rng(11)
    H, L, dh = 2, 260, 128
    lens = rng.permutation(np.r_[1, 2, 3, 17, 33])
    tier_of = [np.concatenate([np.full(lens[0], 1), rng.integers(1, 4, L - lens[0])]).astype(np.int32) for _ in range(H)]
    tier_of[1][:] = np.where(np.arange(L) == 7, 1, np.where(np.arange(L) < 200, 2, 3))         # one token of tier 1
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    for tid, cb in cbs.items():
        C = cb.shape[2]
        if kind == "one":
            cb[:, :, C - 1] = cb[:, :, 0]
        elif kind == "four":
            cb[:, :, C // 4:] = np.tile(cb[:, :, :C // 4], (1, 1, 3, 1))
        else:
            cb[:, :, C // 2:] = cb[:, :, :C // 2]
        if kind == "last_value":
            cb[:, :, C // 2:, -1] = np.nextafter(cb[:, :, C // 2:, -1], np.float32(2))
        if kind == "zero_sign":
            cb[:, :, :, 3] = 0
            cb[:, :, C // 2:, 3] = -0.0
    K = rng.standard_normal((H, L, dh)).astype(np.float32 if fp32 else np.float16)
    log(f"repeated rows {kind} fp32={fp32}")
    r, c, cpu = _codes_and_radii(gpu, rng, K, tier_of, cbs, H, L, dh)
    assert (c == cpu["codes"]).all(), f"{int((c != cpu['codes']).sum())} codes differ"
    assert (r.view(np.uint32) == cpu["r"].view(np.uint32)).all()


@pytest.mark.parametrize("fp32", [False, True])
def test_encode_ties_of_negative_and_zero_similarities(gpu, fp32):
    # every row in one half space and repeated, keys on its other side or
    # orthogonal to all rows: the ranking's threshold lies below zero
    rng = np.random.default_rng(17)
    H, L, dh = 2, 300, 128
    tier_of = [rng.integers(1, 4, L).astype(np.int32) for _ in range(H)]
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    K = np.zeros((H, L, dh))
    for tid, cb in cbs.items():
        G, C, g = cb.shape[1:]
        rows = 0.3 * rng.standard_normal((H, G, C, g)) + 1
        rows[..., g // 2:] = 0
        rows /= np.linalg.norm(rows, axis=-1, keepdims=True)
        cb[:] = rows
        cb[:, :, C // 2:] = cb[:, :, :C // 2]
        for h in range(H):
            for t in np.flatnonzero(tier_of[h] == tid):
                x = 0.2 * rng.standard_normal((G, g)) - 1
                x[:, :g // 2] *= t % 5 > 0
                K[h, t] = (x * 10.0 ** rng.uniform(-3, 2)).reshape(-1)
    K = K.astype(np.float32 if fp32 else np.float16)
    log(f"negative and zero similarities fp32={fp32}")
    r, c, cpu = _codes_and_radii(gpu, rng, K, tier_of, cbs, H, L, dh)
    assert (c == cpu["codes"]).all(), f"{int((c != cpu['codes']).sum())} codes differ"
    assert (r.view(np.uint32) == cpu["r"].view(np.uint32)).all()


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("dh,tier", [(128, 1), (128, 2), (128, 3), (64, 1), (64, 2), (64, 3)])
def test_encode_few_open_codes_of_a_wave(gpu, dh, tier, fp32):
    # runs of 64 tokens (a wave's) of one tier with 0..6 codes that the ranking
    # leaves open: whole and near ties, NaN, infinite and tiny keys; the last
    # page holds one token (torch's M = 1 and small orders)
    rng = np.random.default_rng(100 * tier + dh)
    H, L = 3, 64 * 7 + 1
    cbs = synth.make_codebooks(rng, H, dh, [1, 2, 3])
    cb = cbs[tier]
    G, C, g = cb.shape[1:]
    cb[:, :, C - 1] = cb[:, :, 1]
    K = np.zeros((H, L, dh), np.float64)
    for h in range(H):
        for t in range(L):
            x = cb[h, np.arange(G), rng.integers(2, C - 1, G)] + 0.02 * rng.standard_normal((G, g))
            if t % 64 % 10 < (t // 64 if t < L - 1 else 10) and t % 64 < 10:
                a, b = rng.integers(2, C - 1, 2)
                x = (cb[h, :, 1], cb[h, :, a] + cb[h, :, b] * (1 - 10.0 ** rng.uniform(-7, -4)),
                     1e-20 * x, np.where(rng.random(x.shape) < 0.1, np.inf, x), np.where(rng.random(x.shape) < 0.05, np.nan, x),
                     -cb[h, :, 1])[(t + h) % 6]
            K[h, t] = np.asarray(x).reshape(-1)
    K = K.astype(np.float32 if fp32 else np.float16)
    log(f"few open codes dh={dh} tier={tier} fp32={fp32}")
    _, c, cpu = _codes_and_radii(gpu, rng, K, [np.full(L, tier, np.int32) for _ in range(H)], cbs, H, L, dh)
    assert (c == cpu["codes"]).all(), f"{int((c != cpu['codes']).sum())} codes differ"
