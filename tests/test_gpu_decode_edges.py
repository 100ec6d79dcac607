"""GPU parity at the edges the shared parity suite leaves open.

* Long splits (one split per token over 1,504 records): the record table
  refilled as a split streams, with the second pass of a wide score range.
* Capacity decode (batch 128 x 2 query tokens, top-k 2048, 32,768-record
  contexts) on a pool of 450,000 pages (9.4 GB), so record offsets pass 2^32:
  every token against the oracle, plus pack and reconstruct at the high slots.
* Realistic logit spread (q scaled so logits have a standard deviation of
  about 4) at the batch-1 and batch-64 shapes, checked per (token, head):
  max-abs <= 2e-2 and cosine >= 0.9999 for every row, not only overall.
* Extreme bitmaps (empty words, full words, survivors only in words 0-3 or
  4-7, fully pruned groups with scale byte 105, the reference's tie rows)
  through pack, reconstruct (bit-exact) and the Direct decode
  (scripts/modal/kernels.py:286-287 "bitmap-edges").
* The Direct decode captured in a HIP graph and replayed after q, indices,
  lengths and records change in place (kernels.py:288-289 graph replay).
* The Native store with FP32 input; the batched decode at 4k-128k-token
  contexts (up to 32,768 records).
* FP32-input pack with full-precision mantissas near the threshold and exact
  ties, on many records per wave (the histogram levels of the threshold search).
"""

import numpy as np
import pytest
import torch

import oracle
import remnant
from remnant import _lib
from remnant import synthetic as syn
from test_gpu_parity import (COS_MIN, DEV, OUT_TOL, W1, assert_pool_equal, build_decode_case,
                             check_decode, gpu_pack, oracle_decode, oracle_pack, run_decode)

pytestmark = pytest.mark.gpu


def banner(msg):
    print(f"[gpu-edges] {msg}", flush=True)


def per_row_check(out, ref, lse=None, ref_lse=None):
    """Tolerance per (token, head) row of [.., 512] outputs: the reference's
    attention bar elementwise, |out - ref| <= 0.02 + 0.02 |ref| (output and LSE,
    atol = rtol = 0.02, docs/report.md:20), and cosine >= 0.9999 for every row.
    (A pure max-abs of 0.02 cannot hold for BF16 outputs beyond |8|, where half
    a BF16 ulp is 0.031.)"""
    o = out.reshape(-1, 512).astype(np.float64)
    r = ref.reshape(-1, 512).astype(np.float64)
    excess = (np.abs(o - r) - (OUT_TOL + OUT_TOL * np.abs(r))).max(axis=1)
    assert excess.max() <= 0, f"row {int(excess.argmax())}: beyond atol + rtol by {excess.max()}"
    err = np.abs(o - r).max(axis=1)
    no, nr = np.linalg.norm(o, axis=1), np.linalg.norm(r, axis=1)
    live = (no > 0) | (nr > 0)
    cos = (o * r).sum(axis=1)[live] / np.maximum(no * nr, 1e-300)[live]
    assert cos.min() >= COS_MIN, f"row {int(np.nonzero(live)[0][cos.argmin()])}: cosine {cos.min()}"
    if lse is not None:
        finite = np.isfinite(ref_lse)
        assert np.array_equal(finite, np.isfinite(lse))
        assert (np.abs(lse[finite] - ref_lse[finite]) <=
                OUT_TOL + OUT_TOL * np.abs(ref_lse[finite])).all()
    return float(err.max()), float(cos.min())


# ---- realistic logit spread, per (token, head) ----------------------------------------------

@pytest.mark.parametrize("shape", ["b1", "b64"])
@pytest.mark.parametrize("packed", [True, False], ids=["direct", "native"])
def test_decode_realistic_logit_spread_per_head(shape, packed):
    """q scaled so that the logits q.K / sqrt(512) have std ~4 (unit-RMS rows):
    a few records carry most of each softmax, so the output is far from the
    near-uniform average a small q gives, and every (token, head) row must meet
    the bar on its own."""
    banner(f"decode logit spread {shape} packed={packed}")
    if shape == "b1":
        c = build_decode_case([8192], q_len=1, heads=16, topk=2048, seed=401, packed=packed)
    else:
        ctx = syn.log_uniform_contexts(64, 4096, 32768, 402)
        c = build_decode_case(ctx, q_len=1, heads=16, topk=2048, seed=402, packed=packed)
    c["q"] = (c["q"].float() * 8.0).to(torch.bfloat16)  # N(0, 0.25) * 8 -> std 4
    out, lse = run_decode(c)
    ref, ref_lse = oracle_decode(c)
    # few records dominate each row: the outputs are far from the near-zero
    # average of a near-uniform softmax over independent rows
    assert np.abs(ref).mean() > 0.1
    per_row_check(out, ref, lse, ref_lse)


# ---- extreme bitmaps ---------------------------------------------------------------------------

def extreme_rows(rng):
    """Rows whose top-256 magnitudes fill chosen 64-coordinate groups, with
    names; large values ~N(0,1)*10, the rest tiny."""
    rows, names = [], []

    def groups(full, partial=None):
        x = rng.standard_normal(512).astype(np.float32) * 1e-3
        for g in full:  # magnitudes 20..30, random signs
            x[64 * g:64 * g + 64] = ((20 + 10 * rng.random(64)) *
                                     np.where(rng.random(64) < 0.5, 1, -1)).astype(np.float32)
        if partial:
            for g, idx in partial.items():
                x[64 * g + np.asarray(idx)] = 25.0 + rng.random(len(idx)).astype(np.float32)
        return x

    for full, name in (((0, 1, 2, 3), "words 0-3 only"), ((4, 5, 6, 7), "words 4-7 only"),
                       ((0, 2, 4, 6), "even words"), ((1, 3, 5, 7), "odd words, tail full"),
                       ((7, 0, 1, 2), "tail + 0-2")):
        rows.append(groups(full))
        names.append(name)
    rows.append(groups((0, 1, 2), {3: list(range(63)), 7: [5]}))
    names.append("word 3 has 63, tail 1")
    rows.append(groups((), {g: list(range(32)) for g in range(8)}))
    names.append("half of every word")
    rows.append(groups((), {g: list(range(0, 64, 2)) for g in range(8)}))
    names.append("every other coordinate")
    rows.append(groups((5, 6, 7, 0), {}))
    names.append("tail + 5, 6, 0")
    for r, name in ((np.arange(512), "arange"), (-np.arange(512), "-arange"),
                    (np.zeros(512), "zeros"), (np.ones(512), "ones")):
        rows.append(r.astype(np.float32))
        names.append(name)
    return np.stack(rows), names


def test_extreme_bitmaps_pack_reconstruct_and_decode():
    banner("extreme bitmaps")
    rng = np.random.default_rng(410)
    rows, names = extreme_rows(rng)
    n_ext = rows.shape[0]
    # 128 records: the extreme rows repeated (with sign flips and scales)
    reps = [rows * s for s in (1.0, -1.0, 0.25, 3.0, -7.0, 0.5, 2.0, -1.5, 1.25, -0.75)]
    x = np.concatenate(reps)[:128]
    x = torch.from_numpy(x)
    contexts = [128]
    table = np.array([[1, 0]], np.int32)  # logical record r -> page table[r // 64]
    slots = (table[0, np.arange(128) // 64] * 64 + np.arange(128) % 64).astype(np.int32)
    for dtype in (torch.float32, torch.bfloat16):
        pool = gpu_pack(x.to(dtype), slots, 2)
        ref_pool = oracle_pack(x.to(dtype), slots, 2)
        assert_pool_equal(pool, ref_pool)
        recs = ref_pool.reshape(-1, 328)
        # the intended structures are present: empty and full bitmap words,
        # fully pruned groups (scale byte 105)
        words = recs[slots[:n_ext], 256:320].reshape(n_ext, 8, 8)
        pops = np.unpackbits(words, axis=2).sum(axis=2)
        assert (pops == 0).any() and (pops == 64).any()
        assert (recs[slots[:n_ext], 320:] == 105).any()
        assert pops[0, :4].sum() == 256 and pops[0, 4:].sum() == 0, names[0]
        assert pops[1, 4:].sum() == 256 and pops[1, :4].sum() == 0, names[1]
        # reconstruct every record, with RoPE and without, bit-exact
        freqs = syn.rope_freqs(4 * 128)
        phys = slots.reshape(1, -1)
        raw = np.arange(128, dtype=np.int32).reshape(1, -1)
        lens = np.array([128], np.int32)
        out = torch.empty((128, 512), dtype=torch.bfloat16, device=DEV)
        remnant.unpack_gather_bf16(pool, torch.from_numpy(phys).to(DEV),
                                   torch.from_numpy(raw).to(DEV), torch.from_numpy(lens).to(DEV),
                                   freqs.to(DEV), out, fused_rope=True)
        plain = torch.empty((128, 512), dtype=torch.bfloat16, device=DEV)
        remnant.unpack_gather_bf16(pool, torch.from_numpy(phys).to(DEV), None,
                                   torch.from_numpy(lens).to(DEV), None, plain)
        torch.cuda.synchronize()
        want = oracle.unpack_gather(ref_pool, phys, raw, lens, torch.view_as_real(freqs).numpy())
        assert np.array_equal(syn.bf16_bits(out), want)
        assert np.array_equal(syn.bf16_bits(plain), oracle.unpack_gather(ref_pool, phys, None, lens))
        # Direct decode over all of them (and over the extreme rows alone), with a
        # realistic spread and without
        for q_scale, topk in ((0.5, 128), (6.0, 128), (6.0, n_ext)):
            g = torch.Generator().manual_seed(411)
            q = (torch.randn(1, 2, 16, 512, generator=g) * q_scale).to(torch.bfloat16)
            idx = np.stack([np.random.default_rng(412 + s).permutation(128)[:topk]
                            if topk == 128 else np.arange(topk) for s in range(2)])
            idx = idx.astype(np.int32).reshape(1, 2, topk)
            c = dict(pool=pool, table=table, idx=idx, lens=np.array([topk, topk], np.int32),
                     q=q, sink=torch.randn(16, generator=g), freqs=freqs, contexts=contexts,
                     packed=True)
            out_d, lse_d = run_decode(c)
            ref, ref_lse = oracle_decode(c)
            per_row_check(out_d, ref, lse_d, ref_lse)


# ---- graph replay with changing inputs --------------------------------------------------------

@pytest.mark.parametrize("rope", ["table", "positions"])
@pytest.mark.parametrize("batch,heads,topk", [(8, 64, 64), (1, 16, 2048), (32, 16, 512)])
def test_direct_decode_graph_replay_with_changed_inputs(batch, heads, topk, rope):
    """The decode (and its split combine) captured once; q, indices, lengths
    and the records change in place between replays; every replay equals an
    eager call bit for bit and the oracle within tolerance. The tail rotation
    comes from the table rows or (positions) from the inverse frequencies.
    Splits of one stage (8 x 64 heads, batch 1) and of two stages (32 tokens,
    8 splits: the tail waves beside the MFMA waves)."""
    banner(f"decode graph replay B={batch} H={heads} topk={topk} rope={rope}")
    rng = np.random.default_rng(420 + batch)
    contexts = [int(v) for v in rng.integers(max(topk, 200), 4 * topk + 300, batch)]
    c = build_decode_case(contexts, q_len=1, heads=heads, topk=topk, seed=421 + batch)
    tokens = batch
    q = c["q"].to(DEV)
    bt = torch.from_numpy(c["table"]).to(DEV)
    idx = torch.from_numpy(c["idx"]).to(DEV)
    lens = torch.from_numpy(c["lens"]).to(DEV)
    seq = torch.tensor(contexts, dtype=torch.int32, device=DEV)
    sink = c["sink"].to(DEV)
    rope_kw = ({"rope_inv_freq": syn.rope_inv_freq().to(DEV)} if rope == "positions"
               else {"freqs_cis": c["freqs"].to(DEV)})
    _, need = remnant.get_decode_metadata(tokens, heads, topk)
    ws = torch.zeros(max(need, 1), dtype=torch.uint8, device=DEV)
    out = torch.empty_like(q)
    lse = torch.empty((batch, 1, heads), dtype=torch.float32, device=DEV)
    eager_out = torch.empty_like(q)
    eager_lse = torch.empty_like(lse)

    def call(o, l):
        remnant.remnant_sparse_decode_fwd(q, c["pool"], bt, idx, seqlens=seq, topk_length=lens,
                                          sink=sink, out=o, lse=l, workspace=ws, **rope_kw)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(out, lse)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out, lse)
    torch.cuda.synchronize()
    slots_all = []
    for b, n in enumerate(contexts):
        r = np.arange(n)
        slots_all.append(c["table"][b, r // 64] * 64 + r % 64)
    slots_all = np.concatenate(slots_all).astype(np.int32)
    for it in range(3):
        g = torch.Generator().manual_seed(430 + it)
        q.copy_((torch.randn(q.shape, generator=g) * (0.5 + 2 * it)).to(torch.bfloat16))
        new_idx, new_lens = syn.topk_indices(contexts, 1, topk, seed=431 + it)
        new_lens = np.minimum(new_lens, np.array([topk - 7 * it] * batch, np.int32))
        idx.copy_(torch.from_numpy(new_idx))
        lens.copy_(torch.from_numpy(new_lens))
        # re-pack a third of the records with new latents in place
        pick = np.random.default_rng(432 + it).choice(slots_all.size, slots_all.size // 3,
                                                      replace=False)
        x_new = syn.latents(pick.size, seed=433 + it)
        remnant.pack_rows_fused(x_new.to(DEV), torch.ones(512, device=DEV), 1e-6,
                                torch.from_numpy(slots_all[pick]).to(DEV), c["pool"])
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        call(eager_out, eager_lse)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager_out.view(torch.int16)), it
        assert torch.equal(lse, eager_lse), it
        c["q"] = q.cpu()
        c["idx"] = new_idx
        c["lens"] = new_lens
        ref, ref_lse = oracle_decode(c)
        per_row_check(out.float().cpu().numpy(), ref, lse.cpu().numpy(), ref_lse)


# ---- Native store FP32, batched decode at 4k-128k tokens -----------------------------------

def test_native_store_bit_exact_fp32_input_and_weight():
    banner("native store fp32")
    g = torch.Generator().manual_seed(440)
    n = 768
    x = torch.randn(n, 512, generator=g) * torch.exp(torch.linspace(-3, 3, 512))
    x[::37] *= 1e-30
    x[5::53] = torch.arange(512, dtype=torch.float32) % 5
    w = np.linspace(0.25, 2.0, 512).astype(np.float32)
    slots = np.random.default_rng(440).permutation(n).astype(np.int32)
    slots[::29] = -1
    positions = np.random.default_rng(441).integers(0, 2000, n).astype(np.int32)
    positions[3] = 10_000  # beyond the table: skipped
    freqs = syn.rope_freqs(4 * 2048)
    pool = remnant.LatentPool(n // 64, fmt="native", device=DEV)
    pool.buffer.fill_(0x77)
    remnant.native_store_rows(x.to(DEV), torch.from_numpy(w).to(DEV), 1e-5,
                              torch.from_numpy(slots).to(DEV), torch.from_numpy(positions).to(DEV),
                              freqs.to(DEV), pool)
    torch.cuda.synchronize()
    ref = np.full((n // 64, oracle.NATIVE_PAGE_BYTES), 0x77, np.uint8)
    oracle.native_pack_rows_paged(x.numpy(), w, 1e-5, slots, positions,
                                  torch.view_as_real(freqs).numpy(), ref)
    assert np.array_equal(pool.layer().cpu().numpy(), ref)


@pytest.mark.parametrize("packed", [True, False], ids=["direct", "native"])
def test_decode_batch64_contexts_up_to_128k_tokens(packed):
    """The batched configuration at its full context range: 64 requests of
    4k-128k tokens (1k-32k records), top-k 2048."""
    banner(f"decode B=64 4k-128k packed={packed}")
    ctx = syn.log_uniform_contexts(64, 4096, 131072, 7)
    assert max(ctx) > 16384
    c = build_decode_case(ctx, q_len=1, heads=16, topk=2048, seed=450, packed=packed)
    out, lse = run_decode(c)
    ref, ref_lse = oracle_decode(c)
    per_row_check(out, ref, lse, ref_lse)


# ---- FP32 pack: full-precision mantissas at the threshold ------------------------------------

def test_pack_fp32_full_precision_threshold_mantissas_and_ties():
    """About 100k FP32 records never rounded through BF16, nine or so per wave
    (records 32,768 apart share a wave), each wave's records within 2^+-1 of
    one scale, so the threshold search starts from the previous record's
    exponent. Rows get keys that share the threshold's top 16 bits and differ
    only in mantissa bits 15..0 (the FP32-only histogram levels), and exact
    FP32 ties at the threshold. Checked byte for byte on 8,000 records."""
    banner("pack fp32 full-precision threshold")
    n = 98304 + 4000
    g = torch.Generator().manual_seed(460)
    x = torch.randn(n, 512, generator=g, dtype=torch.float32)
    wave_scale = torch.randint(-20, 21, (32768,), generator=g)
    k = wave_scale[torch.arange(n) % 32768] + torch.randint(-1, 2, (n,), generator=g)
    x = x * torch.pow(2.0, k.float())[:, None]
    xa = x.numpy()
    rng = np.random.default_rng(461)
    # threshold neighbourhoods: the 256th largest magnitude t of a row; put 24
    # keys at t with random low 16 mantissa bits, and 6 exact copies of t
    t_rows = rng.choice(n, n // 3, replace=False)
    mags = np.abs(xa[t_rows])
    t = np.partition(mags, 512 - 256, axis=1)[:, 512 - 256]
    tb = t.view(np.uint32)
    for j in range(24):
        c = rng.integers(0, 512, t_rows.size)
        low = rng.integers(0, 1 << 16, t_rows.size, dtype=np.uint64).astype(np.uint32)
        v = ((tb & 0xFFFF0000) | low).view(np.float32)
        xa[t_rows, c] = np.where(rng.random(t_rows.size) < 0.5, v, -v)
    for j in range(6):
        c = rng.integers(0, 512, t_rows.size)
        xa[t_rows, c] = t * np.where(rng.random(t_rows.size) < 0.5, 1, -1)
    x = torch.from_numpy(xa)
    assert (x.view(torch.int32) & 0xFFFF).ne(0).float().mean() > 0.9  # not BF16 values
    slots = rng.permutation(n).astype(np.int32)
    pages = n // 64 + 1
    gpu = gpu_pack(x, slots, pages)
    pick = np.concatenate([t_rows[:6000], rng.choice(n, 2000, replace=False)])
    ref = oracle_pack(x[pick], slots[pick], pages)
    got = gpu.layer().cpu().numpy().reshape(-1, 328)
    want = ref.reshape(-1, 328)
    bad = np.nonzero((got[slots[pick]] != want[slots[pick]]).any(axis=1))[0]
    assert bad.size == 0, f"{bad.size} records differ, first record {int(pick[bad[0]])}"


# ---- long splits: a split's record table refilled while it streams ------------------------

@pytest.mark.parametrize("topk", [1504, 2208])
@pytest.mark.parametrize("packed", [True, False], ids=["direct", "native"])
def test_decode_long_splits_refilled_table_and_second_pass(packed, topk):
    """128 requests x 2 query tokens x 16 heads (256 token x 16-head blocks, so
    one split per token) at top-k 1504 and 2208: each split streams 47 or 69
    stages of 32 records. Native's 512 table entries are refilled ring-wise as
    the split streams, at both; Packed's table holds 2,048 records and is
    refilled at 2208. Lengths down to 0 end the split inside, at and before the
    table's first wrap; q is scaled so later tiles exceed the first tile's max
    and the split runs a second pass over a rebuilt table. Every row is checked
    against the oracle."""
    banner(f"decode long splits packed={packed} topk={topk}")
    ctx = syn.log_uniform_contexts(128, 6400, 12000, 481)
    if topk > 2048:  # full lists for 16 tokens (the oracle's time)
        ctx = syn.log_uniform_contexts(8, 8900, 12000, 481) + [40] * 120
    c = build_decode_case(ctx, q_len=2, heads=16, topk=topk, seed=481, packed=packed)
    assert remnant.get_decode_metadata(256, 16, topk)[0] == 1
    lens = c["lens"].reshape(-1)
    lens[1:6] = [1000, 513, 512, 31, 0]
    if topk > 2048:
        lens[6:9] = [2049, 2048, 2047]
    c["q"] = (c["q"].float() * 300).to(torch.bfloat16)
    out, lse = run_decode(c)
    ref, ref_lse = oracle_decode(c)
    per_row_check(out, ref, lse, ref_lse)


# ---- capacity decode on a pool above 8 GB ---------------------------------------------------

def test_capacity_decode_b128_next_n2_pool_beyond_4gib_offsets():
    """128 requests x 2 query tokens, top-k 2048 of 32,768-record contexts, on a
    pool of 450,000 pages (9.4 GB): the requests' pages are scattered over the
    whole pool, so most records sit past byte offset 2^32. Every request (all
    256 tokens) is checked against the oracle from a compact copy of the
    requests' pages, for the decode rotating from the table rows and from the
    positions; the pack of two requests' records and a reconstruct of high
    slots are checked byte for byte."""
    banner("capacity decode B=128 x 2, 9.4 GB pool")
    batch, q_len, topk, ctx_records = 128, 2, 2048, 32768
    pool_pages = 450_000
    contexts = [ctx_records] * batch
    table, _ = syn.paged_requests(contexts, 470, pool_pages)
    assert (table.astype(np.int64) * 20992 > (1 << 32)).mean() > 0.4
    pool = remnant.LatentPool(pool_pages, device=DEV)
    w = torch.ones(512, device=DEV)
    tab = torch.from_numpy(table).to(DEV)
    gc = torch.Generator().manual_seed(470)
    sigma = torch.exp(torch.empty(512).uniform_(np.log(0.1), np.log(10.0), generator=gc)).to(DEV)
    r = torch.arange(ctx_records, device=DEV, dtype=torch.int64)

    def request_latents(b):
        g = torch.Generator(device=DEV).manual_seed(1000 + b)
        return (torch.randn(ctx_records, 512, device=DEV, generator=g) * sigma).to(torch.bfloat16)

    for b in range(batch):
        slot = (tab[b, r // 64].to(torch.int64) * 64 + r % 64).to(torch.int32)
        remnant.pack_rows_fused(request_latents(b), w, 1e-6, slot, pool)
    idx, lens = syn.topk_indices(contexts, q_len, topk, seed=471)
    g = torch.Generator().manual_seed(472)
    q = (torch.randn(batch, q_len, 16, 512, generator=g) * 2.0).to(torch.bfloat16)
    sink = torch.randn(16, generator=g)
    freqs = syn.rope_freqs(4 * ctx_records)
    kw = dict(seqlens=torch.tensor(contexts, dtype=torch.int32, device=DEV),
              topk_length=torch.from_numpy(lens).to(DEV), sink=sink.to(DEV))
    outs = {}
    for rope, rkw in (("table", {"freqs_cis": freqs.to(DEV)}),
                      ("positions", {"rope_inv_freq": syn.rope_inv_freq().to(DEV)})):
        outs[rope] = remnant.remnant_sparse_decode_fwd(q.to(DEV), pool, tab,
                                                       torch.from_numpy(idx).to(DEV), **kw, **rkw)
    torch.cuda.synchronize()
    for out, lse in outs.values():
        assert torch.isfinite(out.float()).all() and torch.isfinite(lse).all()
    sample = list(range(batch))
    # compact pool of the requests' pages (1.4 GB), table remapped to it
    pages = torch.from_numpy(table[sample].ravel().astype(np.int64)).to(DEV)
    compact = pool.layer().index_select(0, pages).cpu().numpy()
    ctable = np.arange(len(sample) * table.shape[1], dtype=np.int32).reshape(len(sample), -1)
    sub_lens = lens.reshape(batch, q_len)[sample].ravel()
    ref, ref_lse = oracle.sparse_decode(
        syn.bf16_bits(q[sample]).reshape(len(sample), q_len, 16, 512), compact, True, ctable,
        np.array([ctx_records] * len(sample), np.int32), idx[sample], sub_lens, sink.numpy(),
        torch.view_as_real(freqs).numpy(), 1 / np.sqrt(512))
    for rope, (out, lse) in outs.items():
        banner(f"capacity decode rope={rope}: {2 * len(sample)} tokens against the oracle")
        per_row_check(out[sample].float().cpu().numpy(), ref, lse[sample].cpu().numpy(), ref_lse)
    # the pack at high offsets: two requests' records against the oracle
    for b in (41, 127):
        xs = request_latents(b).float().cpu()
        rows = np.arange(0, ctx_records, 7)  # a seventh of the records
        want = oracle_pack(xs[rows], rows.astype(np.int32), ctx_records // 64)
        i = sample.index(b)
        got = compact[i * 512:(i + 1) * 512].reshape(-1, 328)[rows]
        assert np.array_equal(got, want.reshape(-1, 328)[rows]), b
    # reconstruct from the big pool at the highest slots
    hi_pages = np.argsort(table[sample].ravel())[-64:]
    rows = (hi_pages[:, None] * 64 + np.arange(0, 64, 8)[None]).ravel()  # compact rows
    big = (table[sample].ravel()[hi_pages][:, None].astype(np.int64) * 64 +
           np.arange(0, 64, 8)[None]).ravel()
    assert big.max() * 328 > (1 << 32) and big.max() < (1 << 31)
    out_r = torch.empty((big.size, 512), dtype=torch.bfloat16, device=DEV)
    remnant.unpack_gather_bf16(pool, torch.from_numpy(big.astype(np.int32)).view(1, -1).to(DEV),
                               None, torch.tensor([big.size], dtype=torch.int32, device=DEV),
                               None, out_r)
    torch.cuda.synchronize()
    want = oracle.unpack_gather(compact, rows.astype(np.int32).reshape(1, -1), None,
                                np.array([rows.size], np.int32))
    assert np.array_equal(syn.bf16_bits(out_r), want)
    del pool
    torch.cuda.empty_cache()


def test_native_decode_pool_beyond_4gib_offsets():
    """The Native control decode on a pool of 300,000 pages (11.2 GB): 16
    requests x 2 query tokens, top-k 2048 of 32,768-record contexts, the
    requests' pages scattered over the whole pool so most records sit past byte
    offset 2^32. Every token is checked against the oracle from a compact copy
    of the requests' pages."""
    banner("native decode B=16 x 2, 11.2 GB pool")
    batch, q_len, topk, ctx_records = 16, 2, 2048, 32768
    pool_pages = 300_000
    contexts = [ctx_records] * batch
    table, _ = syn.paged_requests(contexts, 480, pool_pages)
    assert (table.astype(np.int64) * 37376 > (1 << 32)).mean() > 0.5
    pool = remnant.LatentPool(pool_pages, fmt="native", device=DEV)
    w = torch.ones(512, device=DEV)
    tab = torch.from_numpy(table).to(DEV)
    freqs = syn.rope_freqs(4 * ctx_records).to(DEV)
    r = torch.arange(ctx_records, device=DEV, dtype=torch.int64)
    for b in range(batch):
        g = torch.Generator(device=DEV).manual_seed(2000 + b)
        x = torch.randn(ctx_records, 512, device=DEV, generator=g) * 2.0
        slot = (tab[b, r // 64].to(torch.int64) * 64 + r % 64).to(torch.int32)
        remnant.native_store_rows(x, w, 1e-6, slot, r.to(torch.int32), freqs, pool)
    idx, lens = syn.topk_indices(contexts, q_len, topk, seed=481)
    g = torch.Generator().manual_seed(482)
    q = (torch.randn(batch, q_len, 16, 512, generator=g) * 2.0).to(torch.bfloat16)
    sink = torch.randn(16, generator=g)
    out, lse = remnant.native_sparse_decode_fwd(
        q.to(DEV), pool, tab, torch.from_numpy(idx).to(DEV),
        seqlens=torch.tensor(contexts, dtype=torch.int32, device=DEV),
        topk_length=torch.from_numpy(lens).to(DEV), sink=sink.to(DEV))
    torch.cuda.synchronize()
    pages = torch.from_numpy(table.ravel().astype(np.int64)).to(DEV)
    compact = pool.layer().index_select(0, pages).cpu().numpy()
    ctable = np.arange(table.size, dtype=np.int32).reshape(table.shape)
    ref, ref_lse = oracle.sparse_decode(
        syn.bf16_bits(q).reshape(batch, q_len, 16, 512), compact, False, ctable,
        np.array(contexts, np.int32), idx, lens, sink.numpy(), None, 1 / np.sqrt(512))
    per_row_check(out.float().cpu().numpy(), ref, lse.cpu().numpy(), ref_lse)
    del pool
    torch.cuda.empty_cache()


# ---- block-table width: rows looked up in LDS up to 1,024 columns -------------------------

@pytest.mark.parametrize("packed", [True, False], ids=["direct", "native"])
def test_decode_block_table_width(packed):
    """Requests of 1 to 700 records, three query tokens each (a token's request
    by the q_len reciprocal), 14 splits of one stage each, lists that end at and
    beside stage ends. The table as it is, padded to 1,024 columns (looked up in
    LDS) and to 1,025 (looked up in memory): the same bits, and within tolerance
    of the oracle."""
    banner(f"decode block-table width packed={packed}")
    ctx = [700, 1, 64, 65, 333]
    c = build_decode_case(ctx, q_len=3, heads=16, topk=417, seed=487, packed=packed)
    lens = c["lens"].reshape(-1)
    for t, n in ((1, 0), (2, 31), (12, 32), (13, 33), (14, 257)):
        lens[t] = min(n, lens[t])
    out, lse = run_decode(c)
    ref, ref_lse = oracle_decode(c)
    per_row_check(out, ref, lse, ref_lse)
    table = c["table"]
    for width in (1024, 1025):
        c["table"] = np.full((len(ctx), width), -1, np.int32)
        c["table"][:, :table.shape[1]] = table
        got, got_lse = run_decode(c)
        assert np.array_equal(got, out) and np.array_equal(got_lse, lse)


# ---- combine: every count of partials its unrolled loads switch at ------------------------

@pytest.mark.parametrize("topk", [128, 160, 256, 288, 512, 544, 1024, 1056, 2048])
@pytest.mark.parametrize("tokens", [1, 4])
def test_decode_combine_split_counts(tokens, topk):
    """4 to 64 splits of one stage each (one token: the 64-coordinate combine,
    unrolled for 16, 32 and 64 splits) and the same lists over four tokens with
    64 heads (the row combine, unrolled for 4 and 8 splits)."""
    banner(f"decode combine tokens={tokens} topk={topk}")
    c = build_decode_case([2100] * tokens, q_len=1, heads=16 if tokens == 1 else 64, topk=topk,
                          seed=491 + topk, packed=True)
    out, lse = run_decode(c)
    ref, ref_lse = oracle_decode(c)
    per_row_check(out, ref, lse, ref_lse)


# ---- whole and refilled tables around 512 and 2,048 records a split -----------------------

@pytest.mark.parametrize("rope", ["table", "positions"])
@pytest.mark.parametrize("topk", [513, 2048, 2049, 2400])
def test_decode_long_split_table_sizes(topk, rope):
    """One split per token (32 requests x 2 query tokens x 128 heads, 32-head
    workgroups): tables built whole up to 2,048 records,
    refilled beyond, and a second pass (q scaled so that later stages exceed
    the first one's maximum by more than the slack)."""
    banner(f"decode long-split tables topk={topk} {rope}")
    ctx = syn.log_uniform_contexts(32, 2500, 3000, 503)
    for b in (0, 1, 20, 31):  # the requests of the long lists
        ctx[b] = topk + 100
    c = build_decode_case(ctx, q_len=2, heads=128, topk=topk, seed=503, packed=True)
    assert remnant.get_decode_metadata(64, 128, topk)[0] == 1
    c["rope"] = rope
    lens = c["lens"].reshape(-1)
    lens[:] = np.minimum(lens, 40)  # most lists short (the oracle's time)
    lens[[0, 1, 2, 3, 40, 63]] = [topk, 512, 513, 0, topk - 1, topk]
    c["q"] = (c["q"].float() * 300).to(torch.bfloat16)
    out, lse = run_decode(c)
    ref, ref_lse = oracle_decode(c)
    per_row_check(out, ref, lse, ref_lse)


# ---- block table without columns -------------------------------------------------------------

@pytest.mark.parametrize("packed", [True, False], ids=["direct", "native"])
def test_decode_block_table_without_columns(packed):
    """A block table of no columns (max_blocks 0, any stride; through the C ABI,
    since an empty torch tensor has no address) maps no record and none of it is
    read: every list comes out empty, output zero and LSE the sink's."""
    banner(f"decode block table without columns packed={packed}")
    batch, heads, topk = 3, 16, 64
    lib = _lib.load()
    pool = remnant.LatentPool(2, fmt="remnant" if packed else "native", device=DEV)
    q = torch.randn(batch, heads, 512, device=DEV).to(torch.bfloat16)
    idx = torch.arange(topk, dtype=torch.int32, device=DEV).repeat(batch, 1).contiguous()
    sink = torch.randn(heads, device=DEV)
    table = torch.zeros(4, dtype=torch.int32, device=DEV)  # an address; column 0 would be page 0
    need = remnant.get_decode_metadata(batch, heads, topk)[1]
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
    for stride in (0, 1):
        out = torch.full((batch, heads, 512), 7.0, dtype=torch.bfloat16, device=DEV)
        lse = torch.zeros(batch, heads, device=DEV)
        args = [q.data_ptr(), batch, 1, heads, pool.buffer.data_ptr(), 2, table.data_ptr(), stride, 0,
                None, idx.data_ptr(), topk, None, sink.data_ptr()]
        rope = [None, 0, None] if packed else []
        fn = lib.rm_remnant_sparse_decode_fwd if packed else lib.rm_native_sparse_decode_fwd
        assert fn(*args, *rope, 0.1, out.data_ptr(), lse.data_ptr(), ws.data_ptr(), need,
                  torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        assert not out.any()
        # lse = ln(exp(sink)) through base 2: a few FP32 roundings of |sink| < 8
        assert (lse - sink).abs().max() <= 8 * 2.0 ** -22


# ---- short lists in whole tables ----------------------------------------------------------------

@pytest.mark.parametrize("rope", ["table", "positions"])
@pytest.mark.parametrize("heads", [16, 64])
def test_decode_short_lists_in_whole_tables(heads, rope):
    """One split per token at top-k 2048 (256 tokens x 16 heads, 128 x 64 heads in
    32-head workgroups), lists on both sides of each stage and of where the
    set-up writes two slots a thread or all of them (12 stages at 32 heads, 20
    at 16), after lists that filled the table's LDS."""
    banner(f"decode short lists in whole tables heads={heads} {rope}")
    batch, q_len = (128, 2) if heads == 16 else (64, 2)
    topk = 2048
    ctx = syn.log_uniform_contexts(batch, 4 * topk, 4 * topk + 400, 521)
    c = build_decode_case(ctx, q_len=q_len, heads=heads, topk=topk, seed=521, packed=True)
    assert remnant.get_decode_metadata(batch * q_len, heads, topk)[0] == 1
    c["rope"] = rope
    run_decode(c)  # full lists
    lens = c["lens"].reshape(-1)
    edges = [0, 1, 31, 32, 33, 352, 353, 383, 384, 385, 416, 417, 511, 512, 513, 608, 609, 639, 640,
             641, 672, 673]
    lens[:] = np.resize(edges, lens.size)
    out, lse = run_decode(c)
    ref, ref_lse = oracle_decode(c)
    per_row_check(out, ref, lse, ref_lse)


# ---- the splits' shares of a list ---------------------------------------------------------------

def run_split_lse(c, splits):
    """Output, LSE and the split partials' LSEs [tokens, splits, heads] (natural
    log, without the sink) of a decode, from the caller's workspace."""
    batch, q_len, heads = c["q"].shape[:3]
    tokens, topk = batch * q_len, c["idx"].shape[-1]
    got, need = remnant.get_decode_metadata(tokens, heads, topk)
    assert got == splits
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
    kw = dict(seqlens=torch.tensor(c["contexts"], dtype=torch.int32, device=DEV),
              topk_length=torch.from_numpy(c["lens"]).to(DEV), sink=c["sink"].to(DEV),
              workspace=ws)
    fn = remnant.native_sparse_decode_fwd
    if c["packed"]:
        fn = remnant.remnant_sparse_decode_fwd
        kw["freqs_cis"] = c["freqs"].to(DEV)
    out, lse = fn(c["q"].to(DEV), c["pool"], torch.from_numpy(c["table"]).to(DEV),
                  torch.from_numpy(c["idx"]).to(DEV), **kw)
    torch.cuda.synchronize()
    parts = ws.view(torch.float32)[tokens * splits * heads * 512:].cpu().numpy()
    return (out.float().cpu().numpy(), lse.cpu().numpy(),
            parts[:tokens * splits * heads].reshape(tokens, splits, heads) * np.log(2.0))


@pytest.mark.parametrize("packed", [True, False], ids=["direct", "native"])
@pytest.mark.parametrize("batch,q_len,heads,topk,splits",
                         [(5, 3, 16, 417, 14), (8, 2, 64, 317, 4), (32, 2, 16, 2048, 4),
                          (64, 2, 16, 2048, 2), (64, 2, 16, 4160, 2)],
                         ids=["one-stage", "317", "512-a-split", "1024-a-split", "2080-a-split"])
def test_decode_splits_take_consecutive_shares(batch, q_len, heads, topk, splits, packed):
    """Split s of a list of n records in m = ceil(n / 32) stages attends records
    [s c, (s + 1) c) of it, c = 32 ceil(m / splits): its partial's LSE is the
    oracle's over that share alone. Lengths at and beside every stage count at
    which a share moves, in tables of 512 slots, of 2,048 (Packed, two splits of
    1,024) and refilled (Native at 1,024 and both formats at 2,080 records a
    split, two splits)."""
    banner(f"decode split shares {batch}x{q_len}x{heads} topk={topk} packed={packed}")
    # (24 tokens at those lengths, the others' lists short: the oracle's time)
    full = min(batch, -(-24 // q_len))
    ctx = syn.log_uniform_contexts(full, 4 * topk + 128, 4 * topk + 800, 541) + [40] * (batch - full)
    c = build_decode_case(ctx, q_len=q_len, heads=heads, topk=topk, seed=541, packed=packed)
    lens = c["lens"].reshape(-1)
    stages = (topk + 31) // 32
    edges = [0, 1, topk, topk - 1]
    for m in range(1, stages + 1):
        if m % splits in (0, 1) or m in (stages - 1, stages):
            edges += [32 * m - 1, 32 * m, 32 * m + 1]
    edges = np.unique(np.minimum(edges, topk))
    pick = np.linspace(0, edges.size - 1, min(full * q_len, edges.size)).astype(int)
    lens[:full * q_len] = np.resize(edges[pick], full * q_len)
    out, lse, parts = run_split_lse(c, splits)
    ref, ref_lse = oracle_decode(c)
    per_row_check(out, ref, lse, ref_lse)
    lists = c["idx"]
    share = 32 * (-(-(-(-lens // 32)) // splits))
    c["sink"] = None
    for s in range(splits):
        start = np.minimum(s * share, lens)
        count = np.minimum(share, lens - start)
        idx = lists.reshape(lens.size, topk)
        at = np.minimum(start[:, None] + np.arange(max(int(count.max()), 1)), topk - 1)
        c["idx"] = np.take_along_axis(idx, at, axis=1).reshape(batch, q_len, -1).copy()
        c["lens"] = count.astype(np.int32).reshape(np.shape(c["lens"]))
        part_lse = oracle_decode(c)[1].reshape(lens.size, heads)
        empty = count == 0
        assert np.isneginf(parts[empty, s]).all()
        assert np.abs(parts[~empty, s] - part_lse[~empty]).max(initial=0) <= OUT_TOL


# ---- combine: an infinite partial ----------------------------------------------------------------

@pytest.mark.parametrize("tokens,topk,splits", [(1, 96, 3), (1, 544, 17), (1, 1056, 33),
                                                (64, 96, 3), (48, 2048, 6)])
def test_decode_combine_keeps_infinite_partials(tokens, topk, splits):
    """Native records whose coordinates are all 448 * 2^119, below the BF16
    maximum, under q = 0: every weight is 1 and every partial's 448 sums are past
    the FP32 range. The output is infinite there (not NaN: nothing is added for
    the loads past the last split), zero in the tail, the LSE ln(topk)."""
    banner(f"decode combine infinite partials tokens={tokens} topk={topk}")
    pool = remnant.LatentPool(33, fmt="native", device=DEV)
    page = torch.zeros(37376, dtype=torch.uint8)
    page[:36864].view(64, 576)[:, :448] = 0x7E
    page[36864:].view(64, 8)[:, :7] = 127 + 119
    pool.buffer[0] = page.to(DEV)
    q = torch.zeros(tokens, 1, 16, 512, dtype=torch.bfloat16, device=DEV)
    idx = torch.arange(topk, dtype=torch.int32, device=DEV).repeat(tokens, 1, 1).contiguous()
    table = torch.arange(33, dtype=torch.int32, device=DEV).repeat(tokens, 1).contiguous()
    assert remnant.get_decode_metadata(tokens, 16, topk)[0] == splits
    out, lse = remnant.native_sparse_decode_fwd(q, pool, table, idx)
    torch.cuda.synchronize()
    assert (out[..., :448] == float("inf")).all() and not out[..., 448:].any()
    # log2 of the sum and its conversion to base e: a few FP32 roundings of ln(topk) < 8
    assert (lse - np.log(topk)).abs().max() <= 8 * 2.0 ** -22
