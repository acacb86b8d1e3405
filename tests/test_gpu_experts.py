"""GPU parity of the grouped expert products against the CPU oracle.

Decode / verify (xs_native_expert_grouped, the reference's native_expert_grouped contract: q8_1 activations, exact
integer block sums): gate / up within 1e-5 of each row's magnitude, the q8_1 of SwiGLU(gate, up) bit for bit for the
same gate / up, outputs within max|a - b| / max|ref| <= 1e-3 (fp32 accumulate).
Prefill (xs_moe_prefill_experts, f16 MFMA): against a plain PyTorch fp32 reference over the dequantized weights
(xs_iq_dequant_f32 is bit-exact with the reference's dequantizer), max-relative <= 2e-2."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def t2n(t):
    return t.detach().cpu().numpy()


PAIRS = [(8, 8, 1024, 512), (12, 14, 2048, 768), (23, 23, 4096, 1536), (12, 12, 7168, 2048), (8, 8, 7168, 2048),
         (14, 14, 2048, 512), (23, 23, 1024, 256)]


def group_case(n_groups, sizes, n_tok, rng):
    start = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    n = int(start[-1])
    tok = rng.integers(0, n_tok, n).astype(np.int32)
    dst = rng.permutation(n).astype(np.int32)
    return start, tok, dst


@pytest.mark.parametrize("gu,dt,H,F", PAIRS)
def test_native_expert_grouped(xm, xo, gu, dt, H, F):
    rng = np.random.default_rng(H * 7 + F + gu)
    E = 4
    arena, L = xm.build_arena(E, H, F, gu, dt, seed=gu * 31 + H)
    blobs = t2n(arena)
    sizes = [1, 3, 7, 2, 5]                      # groups of 1..7 entries, the last two on the same expert
    experts = [0, 2, 1, 3, 3]
    T = 6
    start, tok, dst = group_case(len(sizes), sizes, T, rng)
    n = int(start[-1])
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16).float()
    xq = xm.quantize_q8_1_rows(x.to(DEV))
    grp_ptr = torch.tensor([arena[e].data_ptr() for e in experts], dtype=torch.int64, device=DEV)
    d_start = torch.from_numpy(start).to(DEV)
    ng = torch.tensor([len(sizes)], dtype=torch.int32, device=DEV)
    scratch = torch.zeros(xm.native_expert_scratch_bytes(n, F), dtype=torch.uint8, device=DEV)
    out = torch.zeros(n, H, device=DEV)
    xm.native_expert_grouped(L, grp_ptr, d_start, ng, torch.from_numpy(dst).to(DEV), torch.from_numpy(tok).to(DEV),
                             len(sizes), n, xq, scratch, out)
    torch.cuda.synchronize()
    ol = xo.layout(gu, dt, H, F)
    want, gate, up, hq = xo.native_expert_grouped(ol, [blobs[e] for e in experts], start, dst, tok, t2n(xq), n,
                                                  want_inner=True)
    fa = (n * F * 4 + 255) & ~255
    sg = t2n(scratch[:n * F * 4].view(torch.float32)).reshape(n, F)
    su = t2n(scratch[fa:fa + n * F * 4].view(torch.float32)).reshape(n, F)
    # the canonical row order is the oracle's: gate / up rows, their SwiGLU q8_1 and the down rows bit for bit
    assert np.array_equal(sg.view(np.uint32), gate.view(np.uint32))
    assert np.array_equal(su.view(np.uint32), up.view(np.uint32))
    hb = t2n(scratch[3 * fa:3 * fa + n * (F // 32) * 36])
    assert np.array_equal(hb, hq)
    assert np.array_equal(t2n(out).view(np.uint32), want.view(np.uint32))
    # and within the reference's float criterion of the exact dot of the dequantized operands
    q, d, _ = xo.q8_1_values(t2n(xq))
    a = (q.astype(np.float64) * d[:, None]).reshape(T, H)
    for e in range(n):
        scale = np.abs(a[tok[e]]).sum() * 0.02 * 4
        assert np.max(np.abs(sg[e] - gate[e])) <= 1e-5 * scale
    status = torch.from_numpy(np.zeros(1, np.int32))
    st = scratch[xm.native_expert_scratch_bytes(n, F) - 256:][:4].view(torch.int32)
    assert int(st[0]) == 0


@pytest.mark.parametrize("gu,dt,H,F", [(12, 14, 2048, 768), (12, 12, 1024, 256), (14, 12, 3072, 512), (14, 14, 2048, 256),
                                       (23, 23, 2048, 512), (23, 8, 1024, 768), (8, 8, 256, 512), (8, 23, 7168, 256)])
def test_native_expert_grouped_many_entries(xm, xo, gu, dt, H, F):
    """Groups large enough for the matrix-core rows: 1 to 70 entries a group (one pass of 16 entries, its edges, and
    passes beyond the four that run side by side), 4 and 8 canonical lanes, every format on either side: the oracle's
    bits, gate and up rows, h and down rows."""
    rng = np.random.default_rng(H + F + gu * 100 + dt)
    arena, L = xm.build_arena(3, H, F, gu, dt, seed=gu + dt)
    blobs = t2n(arena)
    sizes, experts, T = [16, 1, 17, 70, 33, 15], [2, 0, 1, 0, 2, 1], 80
    start, tok, dst = group_case(len(sizes), sizes, T, rng)
    n = int(start[-1])
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16).float()
    xq = xm.quantize_q8_1_rows(x.to(DEV))
    grp_ptr = torch.tensor([arena[e].data_ptr() for e in experts], dtype=torch.int64, device=DEV)
    ng = torch.tensor([len(sizes)], dtype=torch.int32, device=DEV)
    scratch = torch.zeros(xm.native_expert_scratch_bytes(n, F), dtype=torch.uint8, device=DEV)
    out = torch.zeros(n, H, device=DEV)
    print(f"[case] many entries {gu}/{dt} H={H} F={F}", flush=True)
    xm.native_expert_grouped(L, grp_ptr, torch.from_numpy(start).to(DEV), ng, torch.from_numpy(dst).to(DEV),
                             torch.from_numpy(tok).to(DEV), len(sizes), n, xq, scratch, out)
    torch.cuda.synchronize()
    want, gate, up, hq = xo.native_expert_grouped(xo.layout(gu, dt, H, F), [blobs[e] for e in experts], start, dst, tok,
                                                  t2n(xq), n, want_inner=True)
    fa = (n * F * 4 + 255) & ~255
    for off, ref in ((0, gate), (fa, up)):
        got = t2n(scratch[off:off + n * F * 4].view(torch.float32)).reshape(n, F)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(t2n(scratch[3 * fa:3 * fa + n * (F // 32) * 36]), hq)
    assert np.array_equal(t2n(out).view(np.uint32), want.view(np.uint32))
    assert int(scratch[xm.native_expert_scratch_bytes(n, F) - 256:][:4].view(torch.int32)[0]) == 0


def test_grid_groups_same_bits(xm):
    """grid_groups rows of work-groups striding over the groups give the same bits (reference iq_kernels.hpp:85-89)."""
    H, F = 2048, 768
    arena, L = xm.build_arena(6, H, F, 12, 14, seed=5)
    rng = np.random.default_rng(2)
    start, tok, dst = group_case(6, [1, 2, 1, 1, 3, 1], 4, rng)
    n = int(start[-1])
    x = torch.randn(4, H, device=DEV)
    xq = xm.quantize_q8_1_rows(x)
    grp_ptr = torch.tensor([arena[e].data_ptr() for e in range(6)], dtype=torch.int64, device=DEV)
    args = [torch.from_numpy(a).to(DEV) for a in (start, dst, tok)]
    ng = torch.tensor([6], dtype=torch.int32, device=DEV)
    outs = []
    for gg in (0, 1, 4):
        scratch = torch.zeros(xm.native_expert_scratch_bytes(n, F), dtype=torch.uint8, device=DEV)
        out = torch.zeros(n, H, device=DEV)
        xm.native_expert_grouped(L, grp_ptr, args[0], ng, args[1], args[2], 6, n, xq, scratch, out, grid_groups=gg)
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_misaligned_blob_flagged(xm):
    """A blob address off a 16-byte boundary is skipped (never read) and flagged in the scratch status word."""
    H, F = 1024, 512
    arena, L = xm.build_arena(1, H, F, 8, 8, seed=1)
    grp_ptr = torch.tensor([arena[0].data_ptr() + 8], dtype=torch.int64, device=DEV)
    start = torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    zero = torch.zeros(1, dtype=torch.int32, device=DEV)
    ng = torch.ones(1, dtype=torch.int32, device=DEV)
    xq = xm.quantize_q8_1_rows(torch.randn(1, H, device=DEV))
    scratch = torch.zeros(xm.native_expert_scratch_bytes(1, F), dtype=torch.uint8, device=DEV)
    out = torch.zeros(1, H, device=DEV)
    xm.native_expert_grouped(L, grp_ptr, start, ng, zero, zero, 1, 1, xq, scratch, out)
    torch.cuda.synchronize()
    st = scratch[xm.native_expert_scratch_bytes(1, F) - 256:][:4].view(torch.int32)
    assert int(st[0]) == 1


def torch_reference_prefill(xm, arena, L, x, ids, E):
    """fp32 PyTorch reference of the routed products: weights dequantized exactly (xs_iq_dequant_f32), fp32 matmuls,
    h = g / (1 + exp(-g)) * u; returns parts [T*k, H] in routing order."""
    T, H = x.shape
    F = L.n_ff
    k = ids.shape[1]
    parts = torch.zeros(T * k, H, device=DEV)
    flat = ids.reshape(-1)
    for e in torch.unique(flat).tolist():
        rows = torch.nonzero(flat == e).flatten()
        blob = arena[e]
        wg = xm.iq_dequant_f32(L.gu_type, blob[:F * L.gu_row], F * H).reshape(F, H)
        wu = xm.iq_dequant_f32(L.up_type, blob[L.up_off:L.up_off + F * L.up_row], F * H).reshape(F, H)
        wd = xm.iq_dequant_f32(L.d_type, blob[L.down_off:L.down_off + H * L.d_row], H * F).reshape(H, F)
        xs = x[rows // k]
        g = xs @ wg.t().contiguous()
        u = xs @ wu.t().contiguous()
        h = g / (1.0 + torch.exp(-g)) * u
        parts[rows] = h @ wd.t().contiguous()
    return parts


@pytest.mark.parametrize("gu,dt,H,F,T,E", [(12, 14, 2048, 768, 256, 32), (8, 8, 1024, 512, 64, 8),
                                           (23, 23, 4096, 1536, 64, 16), (12, 12, 2048, 512, 5, 16)])
def test_prefill_experts(xm, gu, dt, H, F, T, E):
    k = 8 if E >= 8 else 2
    arena, L = xm.build_arena(E, H, F, gu, dt, seed=gu + H)
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16).float()
    p = 1.0 / torch.arange(1, E + 1, device=DEV, dtype=torch.float32) ** 1.2
    logits = torch.log(p)[None, :] - torch.log(-torch.log(torch.rand(T, E, device=DEV, generator=g)))
    ids, w = xm.router_top10(logits.contiguous(), k)
    r = xm.prefill_route(ids.reshape(-1), k, E, cache_base=arena.data_ptr(), blob=L.bytes, with_ptr=True)
    n = T * k
    cap = min(n, E)
    scratch = torch.zeros(xm.moe_prefill_scratch_bytes(T, n, H, F), dtype=torch.uint8, device=DEV)
    parts = torch.zeros(n, H, device=DEV)
    xm.moe_prefill_experts(L, x, r["src"], r["entry"], r["bounds"], r["n_groups"], r["grp_ptr"], cap, n, scratch,
                           parts)
    torch.cuda.synchronize()
    want = torch_reference_prefill(xm, arena, L, x, ids, E)
    rel = float((parts - want).abs().max() / want.abs().max())
    assert rel <= 2e-2, rel


def test_prefill_experts_saturation_status(xm):
    """xs_moe_prefill_experts flags a value saturated to the f16 range in its scratch's status word
    (xs_moe_prefill_status): clear after a normal call on a zero-filled scratch, bit 8 after a 1e6 activation, and
    xs_moe_status_check raises and clears it."""
    H, F, E, k, T = 1024, 512, 8, 2, 32
    arena, L = xm.build_arena(E, H, F, xm.Q4_K, xm.Q6_K, seed=9)
    g = torch.Generator(device=DEV).manual_seed(9)
    x = torch.randn(T, H, device=DEV, generator=g)
    logits = torch.randn(T, E, device=DEV, generator=g)
    ids, _ = xm.router_top10(logits, k)
    r = xm.prefill_route(ids.reshape(-1), k, E, cache_base=arena.data_ptr(), blob=L.bytes, with_ptr=True)
    n = T * k
    scratch = torch.zeros(xm.moe_prefill_scratch_bytes(T, n, H, F), dtype=torch.uint8, device=DEV)
    status = xm.lib().xs_moe_prefill_status(scratch.data_ptr(), T, n, H, F)
    parts = torch.zeros(n, H, device=DEV)
    for bad in (False, True):
        xb = x.clone()
        if bad:
            xb[3, 7] = 1e6
        xm.moe_prefill_experts(L, xb, r["src"], r["entry"], r["bounds"], r["n_groups"], r["grp_ptr"], min(n, E), n,
                               scratch, parts)
        torch.cuda.synchronize()
        if bad:
            with pytest.raises(xm.XsError, match="f16 range"):
                xm._check(xm.lib().xs_moe_status_check(status, None))
        xm._check(xm.lib().xs_moe_status_check(status, None))   # clear (again)


@pytest.mark.parametrize("T", [2, 3, 4, 5, 16])
@pytest.mark.parametrize("gu,H,F", [(8, 2048, 640), (8, 2048, 1408), (12, 2048, 1408), (8, 4096, 384), (8, 4096, 1536),
                                    (12, 1024, 384), (23, 1024, 640), (23, 4096, 384), (14, 2048, 640)])
def test_q8_0_down_of_several_steps(xm, xo, gu, H, F, T):
    """Q8_0 down rows that the weight stream takes in several steps (F 640: 5, F 1408: 11 at up to 4 tokens), beside
    one-step rows (F 384), more tokens, gate/up rows of four canonical lanes (hidden 1024), Q6_K gate/up rows, which the
    stream does not take, and F 1536, whose rows took two steps before the matrix-core rows: the shared
    expert's rows and the layer's output (hidden 4096: the stream's layers) are the oracle's bits."""
    E, k = 4, 2
    arena, L = xm.build_arena(E, H, F, gu, 8, seed=F + T)
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16).float()
    logits, res = torch.randn(T, E, device=DEV, generator=g), torch.randn(T, H, device=DEV, generator=g)
    print(f"[case] q8_0 down steps gu={gu} H={H} F={F} T={T}", flush=True)
    ol, blobs = xo.layout(gu, 8, H, F), [t2n(arena[e]) for e in range(E)]
    rows, _ = xm.shared_expert_decode(L, arena[1], x)
    assert np.array_equal(t2n(rows).view(np.uint32), xo.shared_expert(ol, blobs[1], t2n(x)).view(np.uint32))
    layer, out = xm.MoeLayer(L, arena, E, k, T), torch.empty_like(res)
    layer(x, logits, res, out)
    want = xo.moe_layer_decode(ol, blobs, k, t2n(x), t2n(logits), t2n(res), n_threads=8)
    assert np.array_equal(t2n(out).view(np.uint32), want.view(np.uint32))
    assert layer.status() == 0


@pytest.mark.parametrize("H,F,sizes", [(256, 512, [1, 16, 17]), (2048, 256, [5, 2]), (4096, 256, [70, 1]), (7168, 512, [16, 3])])
def test_native_expert_grouped_scale_a_block(xm, xo, H, F, sizes):
    """q8_1 rows with a scale of its own in each 32-value block, as a caller's quantizer may give them, for Q8_0 gate/up
    rows: the whole call and its two halves are the oracle's bits (each block's own scale counts)."""
    rng = np.random.default_rng(H + F)
    arena, L = xm.build_arena(2, H, F, 8, 8, seed=H)
    start, tok, dst = group_case(len(sizes), sizes, 20, rng)
    n, experts = int(start[-1]), [i % 2 for i in range(len(sizes))]
    x = rng.standard_normal((20, H)).astype(np.float32) * np.exp(rng.standard_normal((20, H // 32, 1)).repeat(32, 2)
                                                                 .reshape(20, H)).astype(np.float32)
    xq = xo.quantize_q8_1_per32(x)
    dx, d_start, d_tok, d_dst = (torch.from_numpy(v).to(DEV) for v in (xq, start, tok, dst))
    grp_ptr = torch.tensor([arena[e].data_ptr() for e in experts], dtype=torch.int64, device=DEV)
    ng = torch.tensor([len(sizes)], dtype=torch.int32, device=DEV)
    print(f"[case] scale a block H={H} F={F}", flush=True)
    outs = []
    for whole in (True, False):
        scratch = torch.zeros(xm.native_expert_scratch_bytes(n, F), dtype=torch.uint8, device=DEV)
        out = torch.zeros(n, H, device=DEV)
        if whole:
            xm.native_expert_grouped(L, grp_ptr, d_start, ng, d_dst, d_tok, len(sizes), n, dx, scratch, out)
        else:
            xm.native_expert_gate_up(L, grp_ptr, d_start, ng, d_tok, len(sizes), n, dx, scratch)
            xm.native_expert_down(L, grp_ptr, d_start, ng, d_dst, len(sizes), n, scratch, out)
        outs.append(t2n(out))
    want = xo.native_expert_grouped(xo.layout(8, 8, H, F), [t2n(arena[e]) for e in experts], start, dst, tok, xq, n)
    for got in outs:
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("gu,dt,H,F,groups,T", [(12, 14, 1024, 512, 8, 1), (8, 8, 2048, 768, 4, 1), (8, 8, 2048, 768, 5, 1),
                                                (23, 23, 2048, 768, 8, 1), (12, 12, 2048, 768, 8, 1), (12, 12, 4096, 256, 8, 3)])
def test_grouped_of_one_entry_a_group(xm, xo, gu, dt, H, F, groups, T):
    """As many entries as groups by capacity: on either side of the size up to which the lane-per-row kernels take them
    (20 MiB of weights below hidden 4096), and where some groups hold several entries and others are absent all the same:
    the oracle's bits, and a misaligned blob still sets the status word."""
    rng = np.random.default_rng(H + groups)
    arena, L = xm.build_arena(2, H, F, gu, dt, seed=gu + H)
    sizes = [1] * groups if T == 1 else [T] + [1] * (groups - T)      # (fewer groups than the capacity)
    start, tok, dst = group_case(len(sizes), sizes, T, rng)
    n, experts = int(start[-1]), [i % 2 for i in range(len(sizes))]
    assert n == groups
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16).float()
    xq = xm.quantize_q8_1_rows(x.to(DEV))
    ptrs = [arena[e].data_ptr() for e in experts]
    d_start, d_tok, d_dst = (torch.from_numpy(v).to(DEV) for v in (start, tok, dst))
    ng = torch.tensor([len(sizes)], dtype=torch.int32, device=DEV)
    scratch = torch.zeros(xm.native_expert_scratch_bytes(n, F), dtype=torch.uint8, device=DEV)
    out = torch.zeros(n, H, device=DEV)
    print(f"[case] one entry a group {gu}/{dt} H={H} F={F} groups={groups}", flush=True)
    xm.native_expert_grouped(L, torch.tensor(ptrs, dtype=torch.int64, device=DEV), d_start, ng, d_dst, d_tok, groups, n, xq,
                             scratch, out)
    want = xo.native_expert_grouped(xo.layout(gu, dt, H, F), [t2n(arena[e]) for e in experts], start, dst, tok, t2n(xq), n)
    assert np.array_equal(t2n(out).view(np.uint32), want.view(np.uint32))
    word = scratch[xm.native_expert_scratch_bytes(n, F) - 256:][:4].view(torch.int32)
    assert int(word[0]) == 0
    ptrs[0] += 8
    xm.native_expert_grouped(L, torch.tensor(ptrs, dtype=torch.int64, device=DEV), d_start, ng, d_dst, d_tok, groups, n, xq,
                             scratch, out)
    assert int(word[0]) == 1
