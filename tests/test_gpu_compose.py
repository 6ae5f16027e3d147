"""One layer's attention as rLLM composes it (llm/mod.rs:318-354), driven by the C++ batch
builder: a mixed continuous-batching step with prefill chunks that have prior context in the
paged cache plus single-token decode rows, against the oracle pipeline that rLLM's CPU build
runs (scatter -> gather -> repeat_kv -> varlen SDPA for every row)."""
import dataclasses
import math

import numpy as np
import pytest
import torch

from aici_amd import attn, paged
from aici_amd import workloads as W
from aici_amd._lib import HipAttnError
from oracle import refkernels as ref
from tests.common import TOL, make_cache

pytestmark = pytest.mark.gpu


def mixed_step(seed, chunk_priors, chunk_len, n_decode, ctx_lo, ctx_hi, Hq, Hkv, d, dtype, pool, fused_qkv, device,
               paged_prefill=False, bs=16):
    rng = np.random.default_rng(seed)
    g = torch.Generator().manual_seed(seed)
    alloc = paged.BlockAllocator(bs, pool)
    builder = paged.BatchInfoBuilder(bs, 1 << 20, paged_attn_kernel_v=1)
    kc, vc = make_cache(pool, Hkv, d, bs, dtype, fill=float("nan"))  # uninitialised cache
    seqs = []
    sid = 1
    decode_ctx = rng.integers(ctx_lo, ctx_hi + 1, size=n_decode).tolist()
    order = [("chunk", pr) for pr in chunk_priors] + [("decode", c) for c in decode_ctx]
    perm = rng.permutation(len(order))  # interleave: the builder must sort multi-token entries first
    for idx in perm:
        kind, n = order[idx]
        total = n + chunk_len if kind == "chunk" else n
        computed = n if kind == "chunk" else total - 1
        alloc.alloc_seq(sid, total)
        slots = alloc.get_block_idxes(sid, total)
        # the prior context is already in the cache
        kprior = torch.randn((computed, Hkv, d), generator=g).to(dtype)
        vprior = torch.randn((computed, Hkv, d), generator=g).to(dtype)
        ref.reshape_and_cache(kprior, vprior, kc, vc, torch.from_numpy(slots[:computed]))
        builder.sched_out(alloc, sid, rng.integers(0, 1000, size=total).tolist(), computed)
        seqs.append((sid, total, computed))
        sid += 1
    bi = builder.finish()
    T = bi.tokens.numel()
    if fused_qkv:
        assert Hq == Hkv
        qkv = torch.randn((T, 3, Hq, d), generator=g).to(dtype)
        q, k, v = qkv[:, 0], qkv[:, 1], qkv[:, 2]
    else:
        q = torch.randn((T, Hq, d), generator=g).to(dtype)
        k = torch.randn((T, Hkv, d), generator=g).to(dtype)
        v = torch.randn((T, Hkv, d), generator=g).to(dtype)
        qkv = None
    # ---- oracle: the CPU build's route (every row varlen; paged_attn_kernel_v = 0)
    kc_ref, vc_ref = kc.clone(), vc.clone()
    ref.reshape_and_cache(k, v, kc_ref, vc_ref, bi.slot_mapping)
    lens_q = (bi.seqlens_q[1:] - bi.seqlens_q[:-1]).tolist() + [1] * bi.paged_context_lens.numel()
    lens_k = (bi.seqlens_k[1:] - bi.seqlens_k[:-1]).tolist() + bi.paged_context_lens.tolist()
    gather = bi.gather_mapping.tolist()
    for r in range(bi.paged_context_lens.numel()):
        gather += W.slots_for(bi.paged_block_tables[r].tolist(), int(bi.paged_context_lens[r]), bs)
    gm = torch.tensor(gather, dtype=torch.int32)
    gk = torch.empty((len(gather), Hkv, d), dtype=dtype)
    gv = torch.empty_like(gk)
    ref.gather_cached_kv(gk, gv, kc_ref, vc_ref, gm)
    n_rep = Hq // Hkv
    want = ref.varlen_attn(q.float(), ref.repeat_kv(gk, n_rep).float(), ref.repeat_kv(gv, n_rep).float(),
                           W.offsets(lens_q), W.offsets(lens_k), max(lens_q), max(lens_k), 1.0 / math.sqrt(d), True)
    # ---- product: one C-ABI call
    kd, vd = kc.to(device), vc.to(device)
    if fused_qkv:
        qkv_d = qkv.to(device)
        qd, kd_in, vd_in = qkv_d[:, 0], qkv_d[:, 1], qkv_d[:, 2]
    else:
        qd, kd_in, vd_in = q.to(device), k.to(device), v.to(device)
    y = attn.varlen_attn(qd, kd_in, vd_in, bi.to(device), kd, vd, paged_prefill=paged_prefill)
    return y.cpu().reshape(T, Hq, d), want, (kd.cpu(), vd.cpu(), kc_ref, vc_ref), bi


@pytest.mark.parametrize("fused_qkv", [False, True])
def test_mixed_step_phi2_shape_reduced(device, fused_qkv):
    """32 MHA heads of size 80, fp16: 4 chunks of 64 new tokens after 0/100/200/300 cached ones
    plus 20 decode rows, both with contiguous q/k/v and with the fused 3*H*d token stride."""
    y, want, (kc, vc, kc_ref, vc_ref), bi = mixed_step(31, [0, 100, 200, 300], 64, 20, 30, 500, 32, 32, 80,
                                                       torch.float16, 1024, fused_qkv, device)
    assert bi.seqlen_multi == 4 and bi.q_multi == 256 and bi.paged_context_lens.numel() == 20
    assert not torch.isnan(y.float()).any()
    assert (y.float() - want).abs().max().item() <= TOL[torch.float16]
    # the scatter half of the step is bit-exact (NaN-filled slots compare equal as bits)
    assert torch.equal(kc.view(torch.int16), kc_ref.view(torch.int16))
    assert torch.equal(vc.view(torch.int16), vc_ref.view(torch.int16))


def test_mixed_step_gqa_bf16(device):
    y, want, _, bi = mixed_step(32, [0, 17, 640], 200, 33, 1, 900, 32, 8, 128, torch.bfloat16, 2048, False, device)
    assert (y.float() - want).abs().max().item() <= TOL[torch.bfloat16]


@pytest.mark.parametrize("case", ["phi2", "gqa", "all_prefill"])
def test_paged_prefill_route(device, case):
    """The same steps with the multi-token rows reading the cache through block tables
    (hipattn_varlen_attn_paged) instead of a gathered copy."""
    if case == "phi2":
        args, dtype = (31, [0, 100, 200, 300], 64, 20, 30, 500, 32, 32, 80, torch.float16, 1024, True), torch.float16
    elif case == "gqa":
        args, dtype = (32, [0, 17, 640], 200, 33, 1, 900, 32, 8, 128, torch.bfloat16, 2048, False), torch.bfloat16
    else:
        args, dtype = (33, [0, 0, 0], 150, 0, 1, 2, 8, 8, 64, torch.float16, 256, False), torch.float16
    y, want, (kc, vc, kc_ref, vc_ref), bi = mixed_step(*args, device, paged_prefill=True)
    assert bi.multi_block_tables is not None and bi.multi_context_lens.numel() == bi.seqlen_multi
    assert not torch.isnan(y.float()).any()
    assert (y.float() - want).abs().max().item() <= TOL[dtype]
    assert torch.equal(kc.view(torch.int16), kc_ref.view(torch.int16))


@pytest.mark.parametrize("bs", [8, 32])
@pytest.mark.parametrize("paged_prefill", [False, True])
def test_mixed_step_with_8_and_32_token_blocks(device, bs, paged_prefill):
    """The whole composition -- scatter, gather or block tables, prefill rows, decode rows -- on caches of the
    other two block sizes of the reference's matrix."""
    y, want, (kc, vc, kc_ref, vc_ref), bi = mixed_step(35, [0, 17, 640], 200, 33, 1, 900, 32, 8, 128, torch.bfloat16,
                                                       2048 * 16 // bs, False, device, paged_prefill=paged_prefill, bs=bs)
    assert not torch.isnan(y.float()).any()
    assert (y.float() - want).abs().max().item() <= TOL[torch.bfloat16]
    assert torch.equal(kc.view(torch.int16), kc_ref.view(torch.int16))
    assert torch.equal(vc.view(torch.int16), vc_ref.view(torch.int16))


def test_all_prefill_and_all_decode_steps(device):
    y, want, _, bi = mixed_step(33, [0, 0, 0], 150, 0, 1, 2, 8, 8, 64, torch.float16, 256, False, device)
    assert bi.q_multi == 450 and bi.paged_context_lens.numel() == 0
    assert (y.float() - want).abs().max().item() <= TOL[torch.float16]
    y, want, _, bi = mixed_step(34, [], 1, 40, 1, 300, 8, 8, 64, torch.float16, 1024, False, device)
    assert bi.q_multi == 0 and bi.seqlen_multi == 0
    assert (y.float() - want).abs().max().item() <= TOL[torch.float16]


@pytest.mark.parametrize("layout,paged_prefill", [("contiguous", False), ("fused_qkv", False), ("fused_qkv", True)])
def test_config4_full_size_sampled(device, layout, paged_prefill):
    """The benchmark's mixed step at full size: 4 x 512-token chunks after 0/1k/2k/3k cached
    tokens + 120 decode rows with contexts U[1k, 8k], 32 MHA heads, d 80, fp16 -- with contiguous
    q, k, v and with q, k, v as views of one fused [T, 3, H, d] projection (token stride 3*H*d, what
    Phi's layer passes, phi.rs:131-145), the latter also with the multi-token rows reading the cache
    through block tables.  The check (a float64 softmax over the row's gathered context; every row is
    independent) runs on 72 rows: of every chunk its first and last rows and the rows either side of the
    32-, 64-, 96- and 256-row boundaries that the kernels' row blocks and wavefronts cut at, and 24 decode
    rows, the shortest and the longest context among them."""
    rng = np.random.default_rng(4)
    g = torch.Generator().manual_seed(4)
    Hq = Hkv = 32
    d, bs, dtype = 80, 16, torch.float16
    ctxs = rng.integers(1024, 8193, size=120).tolist()
    priors = [0, 1024, 2048, 3072]
    pool = sum((c + 15) // 16 for c in ctxs) + sum((p + 512 + 15) // 16 for p in priors) + 8
    alloc = paged.BlockAllocator(bs, pool)
    builder = paged.BatchInfoBuilder(bs, 1 << 20, 1)
    gd = torch.Generator(device=device).manual_seed(4)
    kd = torch.randn((pool, Hkv, d // 8, bs, 8), generator=gd, dtype=dtype, device=device)
    vd = torch.randn((pool, Hkv, d, bs), generator=gd, dtype=dtype, device=device)
    sid = 1
    for pr in priors:
        alloc.alloc_seq(sid, pr + 512)
        builder.sched_out(alloc, sid, [1] * (pr + 512), pr)
        sid += 1
    for c in ctxs:
        alloc.alloc_seq(sid, c)
        builder.sched_out(alloc, sid, [1] * c, c - 1)
        sid += 1
    bi = builder.finish()
    T = 4 * 512 + 120
    assert bi.tokens.numel() == T and bi.q_multi == 2048
    q = torch.randn((T, Hq, d), generator=g).to(dtype)
    k = torch.randn((T, Hkv, d), generator=g).to(dtype)
    v = torch.randn((T, Hkv, d), generator=g).to(dtype)
    if layout == "fused_qkv":
        qkv = torch.stack([q, k, v], dim=1).to(device)
        qd, kin, vin = qkv[:, 0], qkv[:, 1], qkv[:, 2]
        assert qd.stride(0) == 3 * Hq * d
    else:
        qd, kin, vin = q.to(device), k.to(device), v.to(device)
    y = attn.varlen_attn(qd, kin, vin, bi.to(device), kd, vd, paged_prefill=paged_prefill).reshape(T, Hq, d)
    assert not torch.isnan(y.float()).any()
    kc, vc = kd.cpu(), vd.cpu()  # after the step: holds the new tokens too
    worst = 0.0
    samples = [(512 * i + r, None) for i in range(4) for r in (0, 1, 31, 32, 63, 64, 95, 96, 255, 256, 300, 511)]
    dec_rows = {int(np.argmin(ctxs)), int(np.argmax(ctxs)), *(int(r) for r in rng.choice(120, size=22, replace=False))}
    samples += [(2048 + r, r) for r in sorted(dec_rows)]
    assert len(samples) >= 64
    for row, paged_row in samples:
        if paged_row is None:
            e = row // 512
            lk = priors[e] + 512
            nvis = priors[e] + (row % 512) + 1
            slots = bi.gather_mapping[int(bi.seqlens_k[e]):int(bi.seqlens_k[e]) + lk][:nvis]
        else:
            nvis = int(bi.paged_context_lens[paged_row])
            slots = torch.tensor(W.slots_for(bi.paged_block_tables[paged_row].tolist(), nvis), dtype=torch.int32)
        kk = torch.empty((nvis, Hkv, d), dtype=dtype)
        vv = torch.empty_like(kk)
        ref.gather_cached_kv(kk, vv, kc, vc, slots.to(torch.int32))
        s = torch.einsum("hd,thd->ht", q[row].double(), kk.double()) / math.sqrt(d)
        w = torch.softmax(s, dim=-1)
        want = torch.einsum("ht,thd->hd", w, vv.double())
        worst = max(worst, (y[row].cpu().double() - want).abs().max().item())
    assert worst <= TOL[dtype], worst


STEPS = {  # heads, type, cached tokens in front of each chunk, tokens per chunk, decode rows and their contexts; whether it is one launch
    "gqa": ((32, 8, 128), torch.bfloat16, [0, 640, 1000, 2048], 33, 9, 1, 600, True),                 # pieces; a row block and a row
    "mha": ((32, 32, 80), torch.float16, [255, 0, 256, 257, 1500], 129, 5, 16, 300, True),            # one head a workgroup
    "tile_edges": ((16, 2, 64), torch.float16, [64 * 15 - 32, 64 * 15 - 31, 64 * 15 - 33], 32, 3, 31, 33, True),
    "ratio_2": ((16, 8, 96), torch.bfloat16, [1300, 40], 2, 40, 1, 2000, True),                       # decode shares end inside contexts
    "ratio_3": ((12, 4, 112), torch.float16, [900, 0, 450], 70, 17, 500, 900, True),
    "two_column_groups": ((20, 1, 64), torch.bfloat16, [700, 1], 50, 6, 1, 1500, True),
    "many_chunks": ((8, 2, 128), torch.bfloat16, [300 + i for i in range(70)], 2, 2, 10, 50, True),   # more than a wavefront finds at once
    "chunks_alone": ((32, 8, 128), torch.float16, [3000, 100, 0], 20, 0, 1, 1, True),
    "short": ((32, 8, 128), torch.bfloat16, [0, 100], 20, 4, 10, 200, False),
    "block_8": ((32, 8, 128), torch.bfloat16, [0, 1000], 20, 4, 10, 200, False),
}


def launched(call):
    call()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out = call()
        torch.cuda.synchronize()
    return out, [e.key for e in prof.key_averages()]


@pytest.mark.filterwarnings("ignore:Profiler clears events")
@pytest.mark.parametrize("name", STEPS)
def test_chunks_and_decode_rows_in_one_launch(device, monkeypatch, tuning, name):
    """The launch that holds both kinds of rows against the oracle, against the launches by themselves (a switch that asks for one of
    their kernels), and under an understated bound on the keys."""
    (Hq, Hkv, d), dtype, priors, new, rows, lo, hi, together = STEPS[name]
    bs = 8 if name == "block_8" else 16
    pool = sum(p + new + 2 * bs for p in priors) // bs + rows * (hi // bs + 2) + 8
    routes = {}

    def run(q, k, v, batch, kc, vc, **kw):
        def call():
            return attn_call(q, k, v, batch, kc, vc, **kw)

        y, kernels = launched(call)
        routes["one"] = (y, any("step_merge_kernel" in n for n in kernels))
        short = batch.max_seqlen_k
        batch.max_seqlen_k = max(short - 200, 0)
        routes["understated"] = call()
        batch.max_seqlen_k = short
        tuning("decode_flat", 0)
        y, kernels = launched(call)
        routes["apart"] = (y, any("step_merge_kernel" in n for n in kernels))
        return routes["one"][0]

    attn_call = attn.varlen_attn
    monkeypatch.setattr(attn, "varlen_attn", run)
    y, want, _, _ = mixed_step(40, priors, new, rows, lo, hi, Hq, Hkv, d, dtype, pool, False, device, paged_prefill=bs == 8, bs=bs)
    assert routes["one"][1] == together and not routes["apart"][1]
    for got in (y, *(r.cpu().reshape(y.shape) for r in (routes["understated"], routes["apart"][0]))):
        assert not torch.isnan(got.float()).any()
        assert (got.float() - want).abs().max().item() <= TOL[dtype]


def test_a_captured_step_takes_the_launches_by_themselves(device):
    """A graph holds no pointer into the buffer of the combined launch: replays, with eager steps between them, against the eager result."""
    (Hq, Hkv, d), dtype, priors, new, rows, lo, hi, _ = STEPS["gqa"]
    got = {}

    def run(q, k, v, batch, kc, vc, **kw):
        def call():
            return attn_call(q, k, v, batch, kc, vc, **kw)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            got["eager"] = call()
            attn_call(q[batch.q_multi:], k[batch.q_multi:], v[batch.q_multi:], decode_rows(batch), kc, vc)  # decode's own scratch memory
            side.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                out = call()
            for _ in range(3):
                out.zero_()
                graph.replay()
                assert (out - got["eager"]).abs().max().item() <= TOL[dtype]
                assert torch.equal(call(), got["eager"])
        torch.cuda.current_stream().wait_stream(side)
        return got["eager"]

    def decode_rows(batch):
        alone = dataclasses.replace(batch, q_multi=0, seqlen_multi=0, slot_mapping=batch.slot_mapping[batch.q_multi:].contiguous())
        return alone

    attn_call = attn.varlen_attn
    mp = pytest.MonkeyPatch()
    mp.setattr(attn, "varlen_attn", run)
    try:
        y, want, _, _ = mixed_step(41, priors, new, rows, lo, hi, Hq, Hkv, d, dtype, 2000, False, device)
    finally:
        mp.undo()
    assert (y.float() - want).abs().max().item() <= TOL[dtype]


def random_step(device, heads, dtype, priors, new, contexts, seed=50):
    """A mixed step over caches of random values: (q, k, v, batch on the device, key cache, value cache)."""
    Hq, Hkv, d = heads
    pool = sum(p // 16 + new // 16 + 2 for p in priors) + sum(c // 16 + 1 for c in contexts)
    alloc, builder = paged.BlockAllocator(16, pool), paged.BatchInfoBuilder(16, 1 << 20, 1)
    for sid, (total, computed) in enumerate([(p + new, p) for p in priors] + [(c, c - 1) for c in contexts], 1):
        alloc.alloc_seq(sid, total)
        builder.sched_out(alloc, sid, [1] * total, computed)
    batch = builder.finish().to(device)
    g = torch.Generator(device=device).manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device=device).to(dtype)

    T = batch.tokens.numel()
    return normal(T, Hq, d), normal(T, Hkv, d), normal(T, Hkv, d), batch, normal(pool, Hkv, d // 8, 16, 8), normal(pool, Hkv, d, 16)


@pytest.mark.parametrize("rows,context", [(9, 600), (70, 3000)])  # partitions, flat split
def test_one_eager_step_is_all_that_a_capture_of_it_needs(device, tuning, rows, context):
    """The eager step takes the combined launch, its capture the launches by themselves, on the stream's scratch memory for decode rows."""
    q, k, v, batch, kc, vc = random_step(device, (32, 8, 128), torch.bfloat16, [0, 640, 1000, 2048], 33,
                                         [context - 7 * i for i in range(rows)])

    def call():
        return attn.varlen_attn(q, k, v, batch, kc, vc)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        eager, kernels = launched(call)
        assert any("step_merge_kernel" in n for n in kernels)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = call()
        for _ in range(3):
            out.zero_()
            graph.replay()
            assert (out - eager).abs().max().item() <= TOL[torch.bfloat16]
            assert torch.equal(call(), eager)
        if context < 1024:
            tuning("decode_flat", 0)  # the launches by themselves
            assert torch.equal(call(), out)
    torch.cuda.current_stream().wait_stream(side)


@pytest.mark.parametrize("heads", [1, 4, 16])
@pytest.mark.parametrize("contexts", [[], [5, 40]])
def test_caches_with_other_heads_than_the_keys_are_refused(device, heads, contexts):
    q, k, v, batch, kc, vc = random_step(device, (32, 8, 128), torch.bfloat16, [0, 100], 20, contexts)
    other = k[:, :1].expand(-1, heads, -1)
    with pytest.raises(HipAttnError):
        attn.varlen_attn(q, other, other, batch, kc, vc, cached=True)


def test_a_batch_whose_tables_are_not_those_of_its_rows_is_gathered(device):
    """The first chunk of a batch of two, cut out by hand: the tables still have the rows of both, and may lack their context lengths."""
    q, k, v, batch, kc, vc = random_step(device, (32, 8, 128), torch.bfloat16, [30, 100], 20, [])
    both = attn.varlen_attn(q, k, v, batch, kc, vc)
    n, m = int(batch.seqlens_q[1]), int(batch.seqlens_k[1])
    cut = dict(tokens=batch.tokens[:n], positions=batch.positions[:n], slot_mapping=batch.slot_mapping[:n], q_multi=n, seqlen_multi=1,
               seqlens_q=batch.seqlens_q[:2].contiguous(), seqlens_k=batch.seqlens_k[:2].contiguous(),
               gather_mapping=batch.gather_mapping[:m].contiguous())
    for more in ({}, {"multi_context_lens": None}):
        got = attn.varlen_attn(q[:n], k[:n], v[:n], dataclasses.replace(batch, **cut, **more), kc, vc)
        assert (got - both[:n]).abs().max().item() <= TOL[torch.bfloat16]


@pytest.mark.filterwarnings("ignore:Profiler clears events")
@pytest.mark.parametrize("heads,priors,new,contexts,together", [
    ((40, 8, 112), [900], 1000, [], False),            # 320 workgroups: pieces of their keys would only wait for one another
    ((32, 8, 96), [0], 2000, [60, 300], False),        # 504 of narrow heads beside next to nothing
    ((32, 8, 128), [2000], 4096, [100], False),        # 1032: faster in eight wavefronts, by more than the row is worth
    ((32, 8, 128), [2000], 4096, [3000] * 60, True),   # not by more than these are
    ((12, 4, 112), [800], 300, [], True)])             # 36: seven pieces find compute units without work
def test_which_steps_are_one_launch(device, tuning, heads, priors, new, contexts, together):
    q, k, v, batch, kc, vc = random_step(device, heads, torch.bfloat16, priors, new, contexts)
    got, kernels = launched(lambda: attn.varlen_attn(q, k, v, batch, kc, vc, cached=True))
    assert any("step_merge_kernel" in n for n in kernels) == together
    tuning("decode_flat", 0)  # the launches by themselves
    want = attn.varlen_attn(q, k, v, batch, kc, vc, cached=True)
    assert (got - want).abs().max().item() <= TOL[torch.bfloat16]


def gathered(monkeypatch):
    """attn.varlen_attn on batches without block tables for their chunks: hipattn_varlen_attn, whose gather is counted."""
    calls, inner = [], attn.varlen_attn

    def run(q, k, v, batch, kc, vc, **kw):
        def call():
            return inner(q, k, v, dataclasses.replace(batch, multi_block_tables=None), kc, vc, **kw)

        out, kernels = launched(call)
        calls.append(sum("cache_move" in n for n in kernels))
        return out

    monkeypatch.setattr(attn, "varlen_attn", run)
    return calls


@pytest.mark.filterwarnings("ignore:Profiler clears events")
@pytest.mark.parametrize("name", ["phi2", "phi2_fused", "gqa", "all_prefill", "ratio_2", "ratio_3", "narrow"])
def test_gathered_route_of_16_token_blocks(device, monkeypatch, name):
    args = {"phi2": (31, [0, 100, 200, 300], 64, 20, 30, 500, 32, 32, 80, torch.float16, 1024, False),
            "phi2_fused": (31, [0, 100, 200, 300], 64, 20, 30, 500, 32, 32, 80, torch.float16, 1024, True),
            "gqa": (32, [0, 17, 640], 200, 33, 1, 900, 32, 8, 128, torch.bfloat16, 2048, False),
            "all_prefill": (33, [0, 0, 0], 150, 0, 1, 2, 8, 8, 64, torch.float16, 256, False),
            "ratio_2": (36, [1300, 40], 2, 40, 1, 2000, 16, 8, 96, torch.float16, 3000, False),
            "ratio_3": (37, [900, 0, 450], 70, 17, 500, 900, 12, 4, 112, torch.bfloat16, 1500, False),
            "narrow": (38, [480, 479], 33, 3, 31, 33, 16, 2, 64, torch.bfloat16, 200, False)}[name]
    calls = gathered(monkeypatch)
    y, want, (kc, vc, kc_ref, vc_ref), _ = mixed_step(*args, device)
    assert calls == [2]  # the scatter and the gather
    assert not torch.isnan(y.float()).any()
    assert (y.float() - want).abs().max().item() <= TOL[args[9]]
    assert torch.equal(kc.view(torch.int16), kc_ref.view(torch.int16)) and torch.equal(vc.view(torch.int16), vc_ref.view(torch.int16))


@pytest.mark.filterwarnings("ignore:Profiler clears events")
@pytest.mark.parametrize("layout", ["contiguous", "fused_qkv"])
def test_config4_full_size_gathered(device, monkeypatch, layout):
    calls = gathered(monkeypatch)
    test_config4_full_size_sampled(device, layout, False)
    assert calls == [2]
