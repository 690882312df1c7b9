"""GPU parity of cached decode calls that run the grouped expert kernels (from topk * M * I = 56,000 on): those kernels
copy the misses into their slots, write the victims back and commit the table beside their own work
(csrc/exl3_fill.cuh). Decisions equal the oracle's, every output equals the plain forward on the true blobs bit for bit,
and after the run every slot and every RAM-resident record holds its key's blob."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import cache, synth
from test_gpu_cache import _run, _setup

pytestmark = pytest.mark.gpu
H, I, K, TK = 256, 512, 3, 10                    # noqa: E741


def _check_slots(store, blob_of):
    """Every filled HBM slot holds the blob of the key it is stamped with."""
    torch.cuda.synchronize()
    keys = store.slot_key.cpu().numpy()
    slots = store.slots.view(store.n_slots, -1)
    assert (keys >= 0).any()
    for s in np.nonzero(keys >= 0)[0].tolist():
        want = blob_of(int(keys[s]))
        assert torch.equal(slots[s, :want.numel()], want), f"slot {s} of key {int(keys[s])}"


@pytest.mark.parametrize("M,mode", [(11, "fixed"), (16, "fixed"), (16, "pool"), (16, "ring"), (16, "ring, small"),
                                    (100, "pool")])
def test_cached_grouped_tier(M, mode):
    """3 layers x 128 experts, 150 slots, a 200-record RAM tier, Zipf routing; 110 to 1,000 picks per call. The tier keeps
    fixed records, a record pool, or the victim ring (of 96 slots, and of 4, which drops write-backs)."""
    from pool_checks import check_pool, write_backs
    L, E, S, steps, budget = 3, 128, 150, 40, 200
    ring = {"ring": 96, "ring, small": 4}.get(mode)
    assert M * TK * I >= 56000
    print(f"case cached grouped M={M} {mode}", flush=True)
    ids, w = synth.zipf_trace(20261220 + M, steps, L, E, TK, M=M)
    ids = np.ascontiguousarray(ids.reshape(steps, L, M * TK))
    w = np.ascontiguousarray(w.reshape(steps, L, M * TK))
    co = cache.CacheOracle(L, E, S, ring_cap=1 << 12, budget=budget, age=4, qmax=64, latency=3,
                           **({"victim_ring": ring} if ring else {}))
    orecs, olog = co.run(ids, w)
    store, tier, blobs, ref_ptr = _setup(L, E, S, H, I, K, budget, 64, 4, 3, 1 << 12, 23, pool=mode == "pool",
                                         wb_queue=256, victim_ring=ring)
    recs, bad = _run(store, tier, ids, w, H, check_out_every=1, ref_ptr=ref_ptr, M=M)
    mism = np.nonzero((recs != orecs).any(axis=-1))
    assert mism[0].size == 0, f"first mismatch at step/layer {mism[0][0]}/{mism[1][0]}"
    for n, ((a1, e1), (a2, e2)) in enumerate(zip(tier.decisions, olog)):
        assert a1.tolist() == a2.tolist() and e1.tolist() == e2.tolist(), n
    assert bad == 0
    P = M * TK
    assert recs[:, :, 1].max() > 0 and recs[:, :, 2 + P].sum() > 0        # masked picks and fills happened
    assert write_backs(orecs, P).sum() > 0                                 # and victims were written back
    _check_slots(store, lambda key: blobs[tier.rec_index(key) % tier.src.n])
    if mode == "pool":
        check_pool(store, tier, tier.src, budget, int(write_backs(orecs, P)[:-1].sum()))
    else:
        if ring:
            tier.ring_settle()
            torch.cuda.synchronize()
        for key in np.nonzero(tier.policy.res)[0].tolist():
            want = np.asarray(tier.src.blob_of(tier.rec_index(key)))
            got = np.frombuffer(ctypes.string_at(store.addr(key), want.size), dtype=np.uint8)
            assert np.array_equal(got, want), f"record of key {key}"
    tier.close()


def test_cached_grouped_slots_larger_than_the_blob():
    """Layers at K = 2, 3, 4 in slots of the largest blob, 16 rows x top-8, no tier: a victim may be an expert of another
    bitrate, and leaves as a whole slot. The host record of every expert that enters a slot is overwritten, so the tables
    and outputs are right afterwards only if its write-back brought the bytes home."""
    from exl3xpu import nvtier
    L, E, topk, M, Ks, nd, steps = 3, 96, 8, 16, [2, 3, 4], 4, 30
    print("case cached grouped mixed bitrates", flush=True)
    blob = [nvtier.SyntheticExpertSource(H, I, k, 1, n_distinct=1).blob for k in Ks]
    S = 140
    store = nvtier.TierStore(H, I, 4, E, S, n_layers=L, Ks=Ks)
    keys = [f"model.layers.{li}.mlp" for li in range(L)]
    for k in keys:
        store.add_layer(k)
    srcs = [nvtier.SyntheticExpertSource(H, I, k, 95 + li, n_distinct=nd) for li, k in enumerate(Ks)]
    for key in range(L * E):
        ctypes.memmove(store.addr(key), srcs[key // E].buf[key % nd].ctypes.data, blob[key // E])
    dev = [torch.from_numpy(s.buf).cuda() for s in srcs]
    tables = [torch.tensor([dev[li][e % nd].data_ptr() for e in range(E)], dtype=torch.int64, device="cuda")
              for li in range(L)]
    X = store.X
    ids, w = synth.uniform_trace(96, steps, L, E, topk, M=M)
    x = torch.randn(L, M, H, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).cuda()
    vict = torch.zeros(1 + 2 * E, dtype=torch.int32, device="cuda")
    X.moe_set_victims(vict)
    evicted, wiped = 0, set()
    try:
        for n in range(steps):
            for li in range(L):
                it, wt = torch.from_numpy(ids[n, li]).cuda(), torch.from_numpy(w[n, li]).cuda()
                out = store.forward_cached(keys[li], x[li], it, wt)
                ref = X.moe_forward(x[li], it, wt, tables[li], I, Ks[li], E)
                torch.cuda.synchronize()
                assert torch.equal(out, ref), (n, li)
                v = vict.cpu().numpy()
                home = v[1:1 + 2 * v[0]:2]
                for key in home[home >= 0].tolist():
                    got = np.frombuffer(ctypes.string_at(store.addr(key), blob[key // E]), dtype=np.uint8)
                    assert np.array_equal(got, srcs[key // E].buf[key % nd]), f"write-back of key {key}"
                    wiped.discard(key)
                    evicted += 1
                res = store.slot_key.cpu().numpy()
                for key in set(res[res >= 0].tolist()) - wiped:
                    ctypes.memset(store.addr(key), 0xA5, blob[key // E])
                    wiped.add(key)
    finally:
        X.moe_set_victims(torch.zeros(0, dtype=torch.int32, device="cuda"))
    assert evicted > 0 and wiped
    _check_slots(store, lambda key: dev[key // E][key % nd])


def test_cached_grouped_in_graph_replays():
    """2 layers x 16 rows captured once and replayed over a trace with hits, misses and evictions, with other eager calls
    and synchronizations between the replays: outputs and the whole cache state equal those of a store that runs eagerly."""
    from exl3xpu.moe_offload import ExpertStore
    L, E, S, M, steps = 2, 96, 120, 16, 12
    print("case cached grouped graph", flush=True)
    distinct = [synth.expert_blob(72, e, H, I, K) for e in range(8)]
    stores = []
    for _ in range(2):
        st = ExpertStore(H, I, K, E, S, max_layers=L)
        for li in range(L):
            st.add_layer(li, torch.from_numpy(np.stack([distinct[(li * E + e) % 8] for e in range(E)])))
        stores.append(st)
    ids, w = synth.zipf_trace(97, steps, L, E, TK, M=M)
    ids, w = torch.from_numpy(ids).cuda(), torch.from_numpy(w).cuda()
    x = torch.randn(L, M, H, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    it, wt = ids[0].clone(), w[0].clone()

    def step(st, a, b):
        return [st.forward_cached(li, x[li], a[li], b[li]) for li in range(L)]

    eager = step(stores[0], ids[0].clone(), w[0].clone())
    outs = step(stores[1], it, wt)               # the first call outside the graph
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(eager, outs))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="thread_local"):
        outs = step(stores[1], it, wt)
    fills = 0
    for n in range(1, steps):
        it.copy_(ids[n])
        wt.copy_(w[n])
        graph.replay()
        eager = step(stores[0], ids[n].clone(), w[n].clone())
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(eager, outs)), n
        a, b = stores
        for t in ("slot_of_dev", "slot_key", "slot_last", "tick", "fill_list", "fill_all"):
            assert torch.equal(getattr(a, t), getattr(b, t)), (n, t)
        assert not a.fill_all.any()
        fills += int(a.fill_list[0].item())
    assert fills > 0
    for st in stores:
        _check_slots(st, lambda key: torch.from_numpy(distinct[key % 8]).cuda())
