"""GPU parity of the fused routed-expert FFN (decode M <= 8) against the fp32 CPU oracle.

Tolerances (the bar of the task, on fp32 outputs before the bf16 store):
max-abs <= 2e-2 and rel-L2 <= 1e-3 against the fp32-accumulated oracle; the bf16
output must be within one bf16 rounding step of bf16(oracle) plus the 2e-2 bar.  Against the reference's
own bf16-intermediate route (moe_layer_reference) the distance is that route's
rounding error, ~2-3e-3 rel-L2, asserted <= 6e-3.
"""
import numpy as np
import pytest
import torch

from home_seek_amd import expert_store, fused_moe, ops, synthetic
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

D, I, E, K, SEED = 4096, 2048, 256, 6, 20241


def assert_bf16_close(gb: np.ndarray, rb: np.ndarray, what: str = ""):
    """bf16 result within one bf16 rounding step of bf16(oracle) plus the 2e-2 max-abs bar."""
    bad = np.abs(gb - rb) > np.abs(rb) * 2.0 ** -7 + 2e-2
    assert not bad.any(), (what, np.argwhere(bad)[:5], gb[bad][:5], rb[bad][:5])


def check_close(got_f32: np.ndarray, got_bf16: np.ndarray, ref: np.ndarray, what: str):
    err = got_f32.astype(np.float64) - ref.astype(np.float64)
    rel = np.linalg.norm(err) / np.linalg.norm(ref)
    mx = np.abs(err).max()
    print(f"[{what}] rel-L2 {rel:.3e} max-abs {mx:.3e} (ref rms {np.sqrt(np.mean(ref.astype(np.float64)**2)):.1f})")
    assert rel <= 1e-3 and mx <= 2e-2, (rel, mx)
    assert_bf16_close(orc.bf16_to_f32(got_bf16), orc.bf16_to_f32(orc.f32_to_bf16(ref)), what)


@pytest.fixture(scope="module")
def layer(dev):
    store = expert_store.HbmExpertStore(1, E, D, I, dev, with_shared=True)
    store.fill_synthetic(SEED)
    gate, bias = synthetic.router_weights(SEED, 0, E, D, dev)
    torch.cuda.synchronize()
    return store, gate, bias


_cache = {}


def oracle_expert(eid):
    if eid not in _cache:
        _cache[eid] = orc.gen_fp4_expert(SEED, 0, eid, D, I)
    return _cache[eid]


def oracle_shared():
    if "shared" not in _cache:
        _cache["shared"] = orc.gen_shared_expert(SEED, 0, D, I)
    return _cache["shared"]


def test_store_holds_generated_experts(layer, dev):
    store, _, _ = layer
    views = store.expert_views(0, 5)
    ex = oracle_expert(5)
    assert np.array_equal(views[0].cpu().numpy().view(np.uint8), ex["w1"])
    assert np.array_equal(views[5].view(torch.uint8).cpu().numpy(), ex["w2_scale"])
    sh = store.shared_views(0)
    assert np.array_equal(sh[2].view(torch.uint8).cpu().numpy(), oracle_shared()["w3"])
    assert np.array_equal(sh[5].cpu().numpy(), oracle_shared()["w2_scale"])


def test_single_expert_m1(layer, dev):
    """One routed expert, one token (the reference's CPU M<=8 route)."""
    store, _, _ = layer
    x = synthetic.hidden(SEED, 10, 1, D, dev)
    idx = torch.tensor([[17]], device=dev)
    w = torch.ones(1, 1, device=dev)
    f32 = torch.empty(1, D, dtype=torch.float32, device=dev)
    out, _ = ops.moe_decode(x, idx, w, store.table(0), ops.SCALE_E8M0, None, 10.0, out_f32=f32, d=D, i=I)
    ex = oracle_expert(17)
    ref = orc.expert_ffn_fp32(orc.to_np_bf16(x), ex["w1_bf16"], ex["w3_bf16"], ex["w2_bf16"], 10.0)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), ref, "single expert M=1")


@pytest.mark.parametrize("m", [1, 3, 8])
def test_moe_layer_routed_plus_shared(layer, dev, m):
    store, gate, bias = layer
    x = synthetic.hidden(SEED, 100 + m, m, D, dev)
    idx, w = ops.router_topk(x, gate, bias, K, 1.5)
    f32 = torch.empty(m, D, dtype=torch.float32, device=dev)
    out, _ = ops.moe_decode(x, idx, w, store.table(0), ops.SCALE_E8M0, store.shared_entry(0), 10.0,
                            out_f32=f32, d=D, i=I)
    xn = orc.to_np_bf16(x)
    ridx, rw = orc.router(xn, orc.to_np_bf16(gate), bias.cpu().numpy(), K, 1.5)
    assert np.array_equal(idx.cpu().numpy(), ridx)
    experts = {int(e): oracle_expert(int(e)) for e in np.unique(ridx)}
    ref = orc.moe_layer_fp32(xn, ridx, w.cpu().numpy(), experts, oracle_shared(), 10.0)
    check_close(f32.cpu().numpy(), orc.to_np_bf16(out), ref, f"layer M={m}")
    if m == 3:
        refb = orc.bf16_to_f32(orc.moe_layer_reference(xn, ridx, w.cpu().numpy(), experts, oracle_shared(), 10.0))
        rel = np.linalg.norm(orc.bf16_to_f32(orc.to_np_bf16(out)) - refb) / np.linalg.norm(refb)
        print(f"[layer M=3] rel-L2 vs the reference's bf16-intermediate route: {rel:.3e}")
        assert rel <= 6e-3


def test_deterministic_and_edge_ids(layer, dev):
    store, gate, bias = layer
    x = synthetic.hidden(SEED, 300, 2, D, dev)
    idx = torch.tensor([[4, -1, 9, 300, 4 + 0, 7], [-1, -1, -1, -1, -1, -1]], device=dev)
    idx[0, 4] = 11
    w = torch.tensor([[0.5, 9.0, 0.25, 9.0, 0.125, 0.75], [1.0] * 6], device=dev)
    a, _ = ops.moe_decode(x, idx, w, store.table(0), ops.SCALE_E8M0, None, 10.0, d=D, i=I)
    b, _ = ops.moe_decode(x, idx, w, store.table(0), ops.SCALE_E8M0, None, 10.0, d=D, i=I)
    assert torch.equal(a, b)
    assert torch.count_nonzero(a[1]) == 0  # a token with no valid expert gets zeros
    experts = {e: oracle_expert(e) for e in (4, 9, 11, 7)}
    ref = orc.moe_layer_fp32(orc.to_np_bf16(x[:1]), idx[:1].cpu().numpy(), w[:1].cpu().numpy(), experts, None)
    assert_bf16_close(orc.bf16_to_f32(orc.to_np_bf16(a[:1])), orc.bf16_to_f32(orc.f32_to_bf16(ref)))


def test_fused_moe_forward_with_reference_loaders(layer, dev):
    """FusedMoEFFN.forward with the reference's loader shapes: 6-tuples with fp32
    scales (the engine's GPU tier, engine.py:1260-1271), 3-tuple bf16 weights
    (_load_bf16_deq) and None (absent expert)."""
    store, gate, bias = layer
    moe = fused_moe.FusedMoEFFN(E, I, D, 10.0)
    x = synthetic.hidden(SEED, 400, 3, D, dev)
    idx, w = ops.router_topk(x, gate, bias, K, 1.5)
    ids = sorted(set(idx.cpu().reshape(-1).tolist()))
    absent = ids[0]
    as_bf16 = set(ids[1:4])

    def loader(layer_idx, eid):
        assert layer_idx == 0
        if eid == absent:
            return None
        w1, s1, w3, s3, w2, s2 = store.expert_views(0, eid)
        if eid in as_bf16:
            return ops.fp4_dequant_bf16(w1, s1), ops.fp4_dequant_bf16(w3, s3), ops.fp4_dequant_bf16(w2, s2)
        return w1, s1.to(torch.float32), w3, s3.to(torch.float32), w2, s2.to(torch.float32)

    out = moe.forward(x, idx, w, loader, 0)
    experts = {e: oracle_expert(e) for e in ids if e != absent}
    ref = orc.moe_layer_fp32(orc.to_np_bf16(x), idx.cpu().numpy(), w.cpu().numpy(), experts, None)
    assert_bf16_close(orc.bf16_to_f32(orc.to_np_bf16(out)), orc.bf16_to_f32(orc.f32_to_bf16(ref)))


@pytest.mark.parametrize("form", ["strided", "host", "bf16 scales"])
def test_loader_entries_that_need_work(layer, dev, form):
    """Entries that are not contiguous on the device in a taken scale type give the results of those that are."""
    store, gate, bias = layer
    moe = fused_moe.FusedMoEFFN(E, I, D, 10.0)
    x = synthetic.hidden(SEED, 410, 2, D, dev)
    idx, w = ops.router_topk(x, gate, bias, K, 1.5)

    def ready(layer_idx, eid):
        v = store.expert_views(0, eid)
        return tuple(t if q % 2 == 0 else t.to(torch.float32) for q, t in enumerate(v))

    def other(layer_idx, eid):
        v = ready(layer_idx, eid)
        if form == "strided":
            return tuple(torch.stack((t.view(torch.uint8), t.view(torch.uint8)), dim=-1)[..., 0].view(torch.uint8)
                         if q % 2 == 0 else torch.stack((t, t), dim=-1)[..., 0] for q, t in enumerate(v))
        if form == "host":
            return tuple(t.cpu() for t in v)
        return tuple(t if q % 2 == 0 else t.to(torch.bfloat16) for q, t in enumerate(v))  # (powers of two: exact)

    assert torch.equal(moe.forward(x, idx, w, other, 0), moe.forward(x, idx, w, ready, 0))


@pytest.mark.parametrize("form", ["fp4 loader", "bf16 loader", "shared"])
def test_pinned_weights_refilled_after_the_call(layer, dev, form):
    """The call returns when it has read the host's weights, also behind a busy stream."""
    store = layer[0]
    fp4 = store.expert_views(0, 3)
    src = fp4 if form == "fp4 loader" else tuple(ops.fp4_dequant_bf16(fp4[q], fp4[q + 1]) for q in (0, 2, 4))
    x = synthetic.hidden(SEED, 411, 1, D, dev)
    idx, w = torch.full((1, 1), 3, device=dev), torch.ones(1, 1, device=dev)
    pinned = tuple(torch.empty(t.shape, dtype=t.dtype, pin_memory=True) for t in src)
    busy = torch.randn(4096, 4096, device=dev)

    def call(entry, before):
        def load(layer_idx, eid):
            before()
            return entry
        if form == "shared":
            before()
            return fused_moe.SharedExpertFFN(D, I, 10.0).forward(x[None], *entry)[0]
        return fused_moe.FusedMoEFFN(E, I, D, 10.0).forward(x, idx, w, load, 0)

    def work():
        y = busy
        for _ in range(20):
            y = y @ busy

    want = call(src, lambda: None)
    for t, p in zip(src, pinned):
        p.copy_(t)
    torch.cuda.synchronize()
    got = call(pinned, work)
    for p in pinned:
        p.view(torch.uint8).zero_()
    assert torch.equal(got, want)


def test_expert_table_stays_refused_under_capture(layer, dev, monkeypatch):
    """The table is made from host memory: a graph that copied it would read it again on every replay."""
    entries = [layer[0].expert_views(0, 0)]
    with monkeypatch.context() as mp:
        mp.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        with pytest.raises(RuntimeError, match="capture"):
            ops.expert_table(entries, dev)
    assert int(ops.expert_table(entries, dev)[0, 0]) == entries[0][0].data_ptr()


def test_expert_table_refused_in_a_real_capture(layer, dev):
    """Refused before anything is recorded: the capture goes on and its graph replays."""
    entries = [layer[0].expert_views(0, 0)]
    x, y = torch.ones(4, device=dev), torch.zeros(4, device=dev)
    torch.add(x, 1.0, out=y)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for wait in (True, False):
            with pytest.raises(RuntimeError, match="capture"):
                ops.expert_table(entries, dev, wait=wait)
        torch.add(x, 1.0, out=y)
    for rep in range(3):
        x.fill_(float(rep))
        graph.replay()
        assert y.tolist() == [rep + 1.0] * 4


def test_expert_table_read_on_another_stream(layer, dev):
    """The stream that is current when the table is made is busy; another one reads the table at once."""
    entries = [layer[0].expert_views(0, e) for e in range(E)]
    want = [[t.data_ptr() for t in ent] for ent in entries]
    a = torch.randn(4096, 4096, device=dev)
    torch.cuda.synchronize()
    for _ in range(20):
        a = a @ a
    table = ops.expert_table(entries, dev)
    side = torch.cuda.Stream(dev)
    with torch.cuda.stream(side):
        got = table.clone()
    side.synchronize()
    assert got.tolist() == want


def test_forward_m1_fp4_dict_api(layer, dev):
    store, _, _ = layer
    moe = fused_moe.FusedMoEFFN(E, I, D, 10.0)
    x = synthetic.hidden(SEED, 500, 1, D, dev)
    fp4 = {e: store.expert_views(0, e) for e in (3, 30, 200)}
    rw = {3: 0.7, 30: 0.0, 200: 0.55}
    out = moe.forward_m1_fp4(x, fp4, rw)
    ref = orc.moe_layer_fp32(orc.to_np_bf16(x), np.array([[3, 200]]), np.array([[0.7, 0.55]], np.float32),
                             {3: oracle_expert(3), 200: oracle_expert(200)}, None)
    assert_bf16_close(orc.bf16_to_f32(orc.to_np_bf16(out)), orc.bf16_to_f32(orc.f32_to_bf16(ref)))


def test_shared_expert_ffn_bf16(layer, dev):
    store, _, _ = layer
    sh = oracle_shared()
    w1, w3, w2 = (ops.fp8_dequant_bf16(store.shared_views(0)[2 * q], store.shared_views(0)[2 * q + 1])
                  for q in range(3))
    x = synthetic.hidden(SEED, 600, 2, D, dev)
    out = fused_moe.SharedExpertFFN(D, I, 10.0).forward(x.reshape(1, 2, D), w1, w3, w2)
    ref = orc.expert_ffn_fp32(orc.to_np_bf16(x), sh["w1_bf16"], sh["w3_bf16"], sh["w2_bf16"], 10.0)
    assert_bf16_close(orc.bf16_to_f32(orc.to_np_bf16(out.reshape(2, D))), orc.bf16_to_f32(orc.f32_to_bf16(ref)))


def test_workspace_reuse_across_shapes(layer, dev):
    """Calls of different m share one workspace (largest first): every call must
    still complete its cross-slot reduction (regression: arrival counters
    placed at a shape-dependent offset read stale bytes)."""
    store, gate, bias = layer
    results = {}
    for m in (8, 2, 5, 1):
        x = synthetic.hidden(SEED, 700 + m, m, D, dev)
        idx, w = ops.router_topk(x, gate, bias, K, 1.5)
        out, _ = ops.moe_decode(x, idx, w, store.table(0), ops.SCALE_E8M0, store.shared_entry(0), 10.0, d=D, i=I)
        results[m] = (x, idx, w, out)
    for m, (x, idx, w, out) in results.items():
        experts = {int(e): oracle_expert(int(e)) for e in np.unique(idx.cpu().numpy())}
        ref = orc.moe_layer_fp32(orc.to_np_bf16(x), idx.cpu().numpy(), w.cpu().numpy(), experts, oracle_shared())
        assert_bf16_close(orc.bf16_to_f32(orc.to_np_bf16(out)), orc.bf16_to_f32(orc.f32_to_bf16(ref)), f"m={m}")
