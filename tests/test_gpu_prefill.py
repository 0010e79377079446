"""GPU parity of the prefill grouped GEMM (hsmoe_moe_prefill, m > 8 tokens)
against the fp32 CPU oracle.

Bars (the task's FFN bar, on fp32 outputs): rel-L2 <= 1e-3 and max-abs <= 2e-2
against oracle.moe_layer_fp32; bf16 outputs within one bf16 rounding step of
bf16(oracle) plus 2e-2.  At the full shape (M=512, 256 experts, Zipf(1.1)
routing) the oracle checks a sample of tokens (outputs are per token), and the
whole output is checked against the decode kernels run 8 tokens at a time
(same bar) and for determinism.
"""
import numpy as np
import pytest
import torch

from home_seek_amd import expert_store, fused_moe, ops, synthetic
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SEED, K = 777, 6


def check_close(got_f32, got_bf16, ref, what):
    err = got_f32.astype(np.float64) - ref.astype(np.float64)
    rel = np.linalg.norm(err) / np.linalg.norm(ref)
    mx = np.abs(err).max()
    print(f"[{what}] rel-L2 {rel:.3e} max-abs {mx:.3e}")
    assert rel <= 1e-3 and mx <= 2e-2, (what, rel, mx)
    gb, rb = orc.bf16_to_f32(got_bf16), orc.bf16_to_f32(orc.f32_to_bf16(ref))
    assert not (np.abs(gb - rb) > np.abs(rb) * 2.0 ** -7 + 2e-2).any(), what


class Model:
    def __init__(self, dev, n_experts, d, i, layer=0):
        self.E, self.d, self.i = n_experts, d, i
        self.store = expert_store.HbmExpertStore(1, n_experts, d, i, dev, with_shared=True)
        self.store.fill_synthetic(SEED, [0])
        self._cache = {}

    def expert(self, e):
        if e not in self._cache:
            self._cache[e] = orc.gen_fp4_expert(SEED, 0, e, self.d, self.i)
        return self._cache[e]

    def shared(self):
        if "s" not in self._cache:
            self._cache["s"] = orc.gen_shared_expert(SEED, 0, self.d, self.i)
        return self._cache["s"]

    def oracle(self, x, idx, w, shared=True):
        ids = {int(e) for e in idx.reshape(-1) if 0 <= int(e) < self.E}
        experts = {e: self.expert(e) for e in ids}
        return orc.moe_layer_fp32(orc.to_np_bf16(x), idx, w, experts, self.shared() if shared else None, 10.0)


@pytest.fixture(scope="module")
def small(dev):
    m = Model(dev, 32, 1024, 512)
    torch.cuda.synchronize()
    return m


def run(model, x, idx, w, shared=True, table=None):
    dev = x.device
    f32 = torch.empty(x.shape[0], model.d, dtype=torch.float32, device=dev)
    out, _ = ops.moe_prefill(x, torch.as_tensor(idx, device=dev), torch.as_tensor(w, device=dev),
                             model.store.table(0) if table is None else table, ops.SCALE_E8M0,
                             model.store.shared_entry(0) if shared else None, 10.0, out_f32=f32, i=model.i)
    return out, f32


@pytest.mark.parametrize("m", [9, 40, 100])
def test_small_zipf_routing_matches_oracle(small, dev, m):
    x = synthetic.hidden(SEED, m, m, small.d, dev)
    idx, w = synthetic.zipf_routing(SEED + m, m, small.E, K)
    out, f32 = run(small, x, idx, w)
    ref = small.oracle(x, idx, w)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), ref, f"prefill m={m}")


def test_hot_expert_spans_many_chunks(small, dev):
    """One expert chosen by all 100 tokens (gate/up: chunks of 64 + 36 pairs; down: 4 chunks of <= 32), in varying
    slots."""
    m = 100
    x = synthetic.hidden(SEED, 3, m, small.d, dev)
    idx, w = synthetic.zipf_routing(SEED, m, small.E, K)
    for t in range(m):
        j = t % K
        row = [e for e in idx[t] if e != 7][:K - 1]
        row.insert(j, 7)
        idx[t] = row
    out, f32 = run(small, x, idx, w, shared=False)
    ref = small.oracle(x, idx, w, shared=False)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), ref, "hot expert")


def test_chunk_size_boundaries(small, dev):
    """Buckets of 32, 33, 64, 65 and 97 pairs: gate/up chunks of 32 | 33 | 64 | 64 + 1 | 64 + 33 pairs (the
    64-pair form past 32), down chunks of at most 32; the five experts fill the first slots of their tokens."""
    sizes = {3: 32, 5: 33, 11: 64, 17: 65, 23: 97}
    m = max(sizes.values())
    x = synthetic.hidden(SEED, 7, m, small.d, dev)
    idx, w = synthetic.zipf_routing(SEED + 7, m, small.E, K)
    for t in range(m):
        heads = [e for e in sorted(sizes, key=sizes.get) if t < sizes[e]][:K]
        rest = [int(e) for e in idx[t] if e not in sizes]
        rest += [e for e in range(small.E) if e not in sizes and e not in rest][:K]
        idx[t] = (heads + rest)[:K]
    counts = np.bincount(idx.reshape(-1), minlength=small.E)
    assert all(counts[e] == n for e, n in sizes.items())
    out, f32 = run(small, x, idx, w, shared=False)
    ref = small.oracle(x, idx, w, shared=False)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), ref, "chunk boundaries")


def test_invalid_ids_absent_experts_and_empty_tokens(small, dev):
    m = 20
    x = synthetic.hidden(SEED, 4, m, small.d, dev)
    idx, w = synthetic.zipf_routing(SEED + 4, m, small.E, K)
    idx[0, 1] = -1
    idx[1, 0] = small.E + 5
    idx[2, :] = -1  # no routed expert: the shared expert alone
    idx[3, :] = -1
    table = small.store.table(0).clone()
    table[idx[5, 2]] = 0  # absent expert (loader returned None)
    absent = int(idx[5, 2])
    out, f32 = run(small, x, idx, w, table=table)
    ridx = idx.copy()
    ridx[ridx == absent] = -1
    ref = small.oracle(x, ridx, w)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), ref, "edge ids")
    # no routed and no shared expert -> zeros
    idx2 = np.full((12, K), -1, dtype=np.int64)
    out2, f2 = run(small, x[:12], idx2, w[:12], shared=False)
    assert torch.count_nonzero(f2) == 0 and torch.count_nonzero(out2) == 0


def test_matches_decode_kernels_and_is_deterministic(small, dev):
    m = 64
    x = synthetic.hidden(SEED, 5, m, small.d, dev)
    idx, w = synthetic.zipf_routing(SEED + 5, m, small.E, K)
    out, f32 = run(small, x, idx, w)
    out2, f2 = run(small, x, idx, w)
    assert torch.equal(out, out2) and torch.equal(f32, f2)
    dec = torch.empty_like(f32)
    ti, tw = torch.as_tensor(idx, device=dev), torch.as_tensor(w, device=dev)
    for a in range(0, m, 8):
        ops.moe_decode(x[a:a + 8], ti[a:a + 8], tw[a:a + 8], small.store.table(0), ops.SCALE_E8M0,
                       small.store.shared_entry(0), 10.0, out_f32=dec[a:a + 8], d=small.d, i=small.i)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), dec.cpu().numpy(), "prefill vs decode kernels")


def test_fused_moe_forward_with_fp32_scales_and_bf16_experts(small, dev):
    """FusedMoEFFN.forward at B > 8 with the reference's loader shapes: fp32
    scales, 3-tuple bf16 weights and None; one bf16 expert is chosen by all 40
    tokens (its gate/up chunk of 40 pairs taken as two halves of <= 32)."""
    m = 40
    moe = fused_moe.FusedMoEFFN(small.E, small.i, small.d, 10.0)
    x = synthetic.hidden(SEED, 6, m, small.d, dev)
    idx, w = synthetic.zipf_routing(SEED + 6, m, small.E, K)
    ids = sorted({int(e) for e in idx.reshape(-1)})
    absent, as_bf16 = ids[0], set(ids[1:4])
    hot = ids[1]
    for t in range(m):
        if hot not in idx[t]:
            idx[t, t % K] = hot

    def loader(layer_idx, eid):
        if eid == absent:
            return None
        w1, s1, w3, s3, w2, s2 = small.store.expert_views(0, eid)
        if eid in as_bf16:
            return ops.fp4_dequant_bf16(w1, s1), ops.fp4_dequant_bf16(w3, s3), ops.fp4_dequant_bf16(w2, s2)
        return w1, s1.to(torch.float32), w3, s3.to(torch.float32), w2, s2.to(torch.float32)

    out = moe.forward(x, torch.as_tensor(idx, device=dev), torch.as_tensor(w, device=dev), loader, 0)
    ridx = idx.copy()
    ridx[ridx == absent] = -1
    ref = small.oracle(x, ridx, w, shared=False)
    gb, rb = orc.bf16_to_f32(orc.to_np_bf16(out)), orc.bf16_to_f32(orc.f32_to_bf16(ref))
    assert not (np.abs(gb - rb) > np.abs(rb) * 2.0 ** -7 + 2e-2).any()


def test_full_shape_m512_zipf(dev):
    """Config shape: M=512, D=4096, I=2048, 256 experts, Zipf(1.1) top-6 + shared."""
    model = Model(dev, 256, 4096, 2048)
    m = 512
    x = synthetic.hidden(SEED, 512, m, model.d, dev)
    idx, w = synthetic.zipf_routing(1234, m, model.E, K)
    counts = np.bincount(idx.reshape(-1), minlength=model.E)
    print(f"touched experts {np.count_nonzero(counts)}, max tokens/expert {counts.max()}")
    out, f32 = run(model, x, idx, w)
    sample = [0, 1, 2, 255, 256, 400, 510, 511]
    ref = model.oracle(x[sample], idx[sample], w[sample])
    check_close(f32[sample].cpu().numpy(), orc.to_np_bf16(out[sample]), ref, "M=512 sample")
    dec = torch.empty_like(f32)
    ti, tw = torch.as_tensor(idx, device=dev), torch.as_tensor(w, device=dev)
    for a in range(0, m, 8):
        ops.moe_decode(x[a:a + 8], ti[a:a + 8], tw[a:a + 8], model.store.table(0), ops.SCALE_E8M0,
                       model.store.shared_entry(0), 10.0, out_f32=dec[a:a + 8], d=model.d, i=model.i)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), dec.cpu().numpy(), "M=512 vs decode kernels")


@pytest.mark.parametrize("m,k", [(96, 8), (97, 8), (128, 6), (153, 5), (154, 5), (513, 2)])
def test_group_kernel_either_side_of_768_pairs(small, dev, m, k):
    """Up to 768 pairs are grouped by 256 threads, more by 1024: rows as of calls of 64 tokens, bit for bit
    (a pair's sums do not depend on its chunk)."""
    x = synthetic.hidden(SEED, 60 + m, m, small.d, dev)
    g = torch.Generator(dev).manual_seed(m)
    idx = torch.stack([torch.randperm(small.E + 2, generator=g, device=dev)[:k] - 1 for _ in range(m)])  # (-1, E: none)
    w = torch.rand(m, k, device=dev, generator=g)
    table, shared = small.store.table(0), small.store.shared_entry(0)
    whole, parts = (torch.empty(m, small.d, dtype=torch.float32, device=dev) for _ in range(2))
    ops.moe_prefill(x, idx, w, table, ops.SCALE_E8M0, shared, 10.0, out_f32=whole, i=small.i)
    for a in range(0, m, 64):
        ops.moe_prefill(x[a:a + 64], idx[a:a + 64], w[a:a + 64], table, ops.SCALE_E8M0, shared, 10.0,
                        out_f32=parts[a:a + 64], i=small.i)
    assert torch.equal(whole, parts)


@pytest.fixture(scope="module")
def odd(dev):
    m = Model(dev, 9, 1024, 1536)  # 6 K-chunks in the down pass: its last read of scales is a half one
    torch.cuda.synchronize()
    return m


def wide_rule(pairs, n_exp, i, shared):
    """Which calls take the 32-row kernels (hsmoe_moe_prefill's rule)."""
    return pairs > 32 if n_exp == 1 else pairs >= (24 if shared else 32) * n_exp and pairs * i >= 12288 * 1024


def entries_of(model, n_exp, kind):
    """The first n_exp experts in one of the weight formats."""
    entries = []
    for e in range(n_exp):
        w1, s1, w3, s3, w2, s2 = model.store.expert_views(0, e)
        if kind == "bf16":
            entries.append(tuple(ops.fp4_dequant_bf16(a, b) for a, b in ((w1, s1), (w3, s3), (w2, s2))))
        elif kind == "f32":
            entries.append((w1, s1.to(torch.float32), w3, s3.to(torch.float32), w2, s2.to(torch.float32)))
        else:
            entries.append((w1, s1, w3, s3, w2, s2))
    return entries


@pytest.mark.parametrize("kind", ["e8m0", "f32", "bf16"])
@pytest.mark.parametrize("n_exp,m,shared", [(1, 33, False), (1, 500, False), (1, 1089, True), (1, 1601, False),
                                            (2, 40, True), (9, 131, True)])
def test_wide_kernels_every_format(odd, dev, kind, n_exp, m, shared):
    """One expert on the 32-row kernels in every weight format: chunks of 32 pairs (33, 500 and 1089) and of 64
    (1601, the shared expert's) with ragged ends.  The calls of 2 and 9 experts are below the line of those
    kernels (wide_rule): the same formats on the 16-row ones."""
    assert wide_rule(m * (1 if n_exp < 3 else 2), n_exp, odd.i, shared) == (n_exp == 1)
    k = 1 if n_exp < 3 else 2
    entries = entries_of(odd, n_exp, kind)
    table = ops.expert_table(entries, dev)
    x = synthetic.hidden(SEED, 40 + m, m, odd.d, dev)
    idx = np.stack([(np.arange(m) * (j + 1) + j) % min(n_exp, 7) for j in range(k)], axis=1).astype(np.int64)
    if n_exp == 9:
        idx[:5, 0], idx[5:38, 1] = 7, 8  # a small expert and one of 33 pairs
    if k == 2:
        idx[idx[:, 0] == idx[:, 1], 1] = -1
    w = np.linspace(0.2, 1.1, m * k, dtype=np.float32).reshape(m, k)
    f32 = torch.empty(m, odd.d, dtype=torch.float32, device=dev)
    out, _ = ops.moe_prefill(x, torch.as_tensor(idx, device=dev), torch.as_tensor(w, device=dev), table,
                             ops.SCALE_F32 if kind == "f32" else ops.SCALE_E8M0,
                             odd.store.shared_entry(0) if shared else None, 10.0, out_f32=f32, i=odd.i)
    sample = np.unique(np.r_[0:m:7, 30:34, m - 3:m] % m)
    ref = odd.oracle(x[sample], idx[sample], w[sample], shared=shared)
    check_close(f32[sample].cpu().numpy(), orc.to_np_bf16(out[sample]), ref, f"wide {kind} E={n_exp} m={m}")


@pytest.mark.parametrize("kind", ["e8m0", "f32", "bf16"])
@pytest.mark.parametrize("n_exp,m,shared", [(9, 4099, True), (9, 4099, False), (7, 4107, True), (2, 4098, False)])
def test_wide_kernels_several_experts(odd, dev, kind, n_exp, m, shared):
    """The 32-row kernels in calls of several experts: chunks placed by chunk (9 experts) and by row block (7 and 2),
    small experts beside them (5 and 32 pairs: the 16-row kernels), chunks of 33, 64 and 64 + 1 pairs and long ones,
    an absent expert, invalid ids, the shared expert's FP8 chunks before the routed ones."""
    k = 2
    assert wide_rule(m * k, n_exp, odd.i, shared)
    entries = entries_of(odd, n_exp, kind)
    idx = np.stack([np.arange(m) % 2, np.full(m, -1)], axis=1).astype(np.int64)
    few = 0  # tokens below this select experts of at most 32 pairs only
    if n_exp > 2:
        entries[3] = None
        counts = {4: 5, 5: 32, 6: 33} if n_exp == 7 else {4: 5, 5: 32, 6: 33, 7: 64, 8: 65}
        few = counts[4] + counts[5]
        idx[:few, 0], idx[:few, 1] = np.repeat([4, 5], [5, 32]), [-1, n_exp, 3] * 12 + [-1]
        at = few
        for e in sorted(counts)[2:]:
            idx[at:at + counts[e], 1] = e
            at += counts[e]
        idx[at:at + 2000, 1] = 2
        assert np.bincount(idx[idx >= 0], minlength=n_exp)[4:n_exp].tolist() == list(counts.values())
    else:
        idx[:, 1] = 1 - idx[:, 0]
        idx[::5, 1] = 2  # (no such expert)
    w = np.linspace(0.2, 1.1, m * k, dtype=np.float32).reshape(m, k)
    table, scale = ops.expert_table(entries, dev), ops.SCALE_F32 if kind == "f32" else ops.SCALE_E8M0
    sh = odd.store.shared_entry(0) if shared else None
    x = synthetic.hidden(SEED, 70 + m, m, odd.d, dev)
    ti, tw = torch.as_tensor(idx, device=dev), torch.as_tensor(w, device=dev)
    whole, parts = (torch.empty(m, odd.d, dtype=torch.float32, device=dev) for _ in range(2))
    out, _ = ops.moe_prefill(x, ti, tw, table, scale, sh, 10.0, out_f32=whole, i=odd.i)
    for a in range(0, m, 512):  # below the line: the 16-row kernels
        assert not wide_rule(512 * k, n_exp, odd.i, shared)
        ops.moe_prefill(x[a:a + 512], ti[a:a + 512], tw[a:a + 512], table, scale, sh, 10.0,
                        out_f32=parts[a:a + 512], i=odd.i)
    # the two forms add in another order, and the small experts' pairs keep the 16-row one
    assert not torch.equal(whole[few:], parts[few:])
    if not shared:
        assert torch.equal(whole[:few], parts[:few])
    what = f"wide {kind} E={n_exp} m={m} shared={shared}"
    check_close(whole.cpu().numpy(), orc.to_np_bf16(out), parts.cpu().numpy(), what + " vs 16-row kernels")
    sample = np.unique(np.r_[0:few:6, few:few + 300:11, m - 3:m] % m)
    taken = idx[sample].copy()
    taken[(taken >= n_exp) | ((taken == 3) & (n_exp > 2))] = -1
    check_close(whole[sample].cpu().numpy(), orc.to_np_bf16(out[sample]),
                odd.oracle(x[sample], taken, w[sample], shared=shared), what)
