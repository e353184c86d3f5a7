"""HIP-graph capture of a full decode step (writer + split prep + packed decode).

Serving captures the decode step in a graph (deployment/serve.py:164) with a
padded batch: padding rows use slot 0, which must never claim a window row
(mla_fused_writer.py:41-43), and the decode scratch is sized for the captured
batch (rolaq_sglang.patch:62-111). The captured step is replayed over several
decode steps, with this program's own eager work (new inputs copied into the
static buffers) between replays; every replay must leave the pool and the
output exactly as the same step run eagerly on a twin pool, and the replayed
outputs of the live rows must match the oracle's dequantize-then-attention over
the rows the replays wrote (rtol 2e-2 / atol 2e-3).
"""

import math

import numpy as np
import pytest
import torch

from oracle import attention
from mla_kv_quant_amd import PackedMLAPool, synth, writer
from mla_kv_quant_amd.decode import packed_mla_decode_gf_fwd, prepare_gf_splits
from tests.helpers import gpu_pool_to_oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_captured_decode_step_replays_match_eager():
    D, R, H, P, W, layers = 512, 64, 16, 4, 16, 2
    lengths0 = [40, 100, 7]
    nreq, Bg, steps, size, max_splits = len(lengths0), len(lengths0) + 1, 5, 512, 8
    rots = [synth.make_rotation(D, 300 + i) for i in range(layers)]

    def make_pool():
        return PackedMLAPool(size, layers, D, R, 8, P, W, device=DEV, rotations=rots)

    pools = {"graph": make_pool(), "eager": make_pool()}
    base = [1 + 150 * b for b in range(nreq)]  # request b owns slots base_b .. base_b + 149
    for li in range(layers):
        for b, L in enumerate(lengths0):
            loc = torch.arange(base[b], base[b] + L, device=DEV)
            x = synth.make_latent(L, D, 5, seed=10 * li + b).to(DEV)
            pe = synth.make_normal((L, R), 20 * li + b).to(DEV)
            for p in pools.values():
                writer.write_prefill(p, li, loc, x, pe, torch.arange(L, device=DEV), torch.full((L,), L, device=DEV),
                                     torch.full((L,), b + 1, device=DEV))

    sm = 1 / math.sqrt(192)
    maxtok = sum(lengths0) + nreq * steps + 1
    st = {  # static inputs of the captured step
        "loc": torch.zeros(Bg, dtype=torch.int64, device=DEV),
        "seq": torch.ones(Bg, dtype=torch.int64, device=DEV),
        "req": torch.zeros(Bg, dtype=torch.int64, device=DEV),
        "ckv": torch.zeros(layers, Bg, D, dtype=torch.bfloat16, device=DEV),
        "kpe": torch.zeros(layers, Bg, R, dtype=torch.bfloat16, device=DEV),
        "q": torch.zeros(layers, Bg, H, D + R, dtype=torch.bfloat16, device=DEV),
        "indptr": torch.zeros(Bg + 1, dtype=torch.int32, device=DEV),
        "indices": torch.zeros(maxtok, dtype=torch.int32, device=DEV),
        "ns": torch.full((Bg,), 4, dtype=torch.int32, device=DEV),
    }
    quant, merge = torch.empty_like(st["ns"]), torch.empty_like(st["ns"])
    outs = {k: {"logits": torch.empty(Bg, H, max_splits + 1, D, device=DEV),
                "lse": torch.empty(Bg, H, max_splits + 1, device=DEV),
                "o": torch.zeros(layers, Bg, H, D, dtype=torch.bfloat16, device=DEV)} for k in pools}

    def set_inputs(s):
        lens = [L + s + 1 for L in lengths0]
        loc = [base[b] + lens[b] - 1 for b in range(nreq)] + [0]          # padding row -> slot 0
        seq = lens + [1]
        req = [b + 1 for b in range(nreq)] + [0]
        idx = np.concatenate([np.arange(base[b], base[b] + lens[b]) for b in range(nreq)] + [np.zeros(1)])
        ptr = np.concatenate([[0], np.cumsum(lens + [1])])
        st["loc"].copy_(torch.tensor(loc))
        st["seq"].copy_(torch.tensor(seq))
        st["req"].copy_(torch.tensor(req))
        st["indices"][: len(idx)].copy_(torch.from_numpy(idx.astype(np.int32)))
        st["indptr"].copy_(torch.from_numpy(ptr.astype(np.int32)))
        st["ckv"].copy_(synth.make_latent(layers * Bg, D, 5, seed=500 + s).view(layers, Bg, D))
        st["kpe"].copy_(synth.make_normal((layers, Bg, R), 600 + s))
        st["q"].copy_(synth.make_normal((layers, Bg, H, D + R), 700 + s, std=2 / (sm * math.sqrt(D + R))))

    def step(pool, out):
        pool.set_window_meta(True, st["seq"], st["req"])
        prepare_gf_splits(st["ns"], quant, merge)
        for li in range(layers):
            assert writer.try_fast_decode_store(pool, li, st["loc"], st["ckv"][li], st["kpe"][li])
            packed_mla_decode_gf_fwd(st["q"][li], out["o"][li], pool, li, st["indptr"], st["indices"], st["ns"],
                                     max_splits, out["logits"], out["lse"], sm, seq_lens=st["seq"],
                                     req_pool_indices=st["req"])

    set_inputs(0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(pools["graph"], outs["graph"])  # warm-up (caches the bf16 rotations)
    torch.cuda.current_stream().wait_stream(side)
    step(pools["eager"], outs["eager"])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(pools["graph"], outs["graph"])

    for s in range(steps):
        set_inputs(s)
        graph.replay()
        step(pools["eager"], outs["eager"])
        torch.cuda.synchronize()
        og, oe = outs["graph"]["o"], outs["eager"]["o"]
        assert torch.isfinite(og[:, :nreq].float()).all()
        assert torch.equal(og, oe), f"replay {s}: output differs from the eager step"
        pg, pe_ = pools["graph"], pools["eager"]
        for li in range(layers):
            for name in ("c_codes", "c_params", "rope_buf", "hp_c"):
                assert torch.equal(getattr(pg, name)[li], getattr(pe_, name)[li]), (s, li, name)
        assert torch.equal(pg.hp_row_of_slot, pe_.hp_row_of_slot)
        assert torch.equal(pg.hp_owner_of_row, pe_.hp_owner_of_row)
        # slot 0 (graph padding) never claims a window row
        assert int(pg.hp_row_of_slot[0]) == -1
        # the replayed outputs of the live rows against the oracle's
        # dequantize-then-attention over the rows the replays wrote
        lens = [L + s + 1 for L in lengths0]
        slots = [np.arange(base[b], base[b] + lens[b]) for b in range(nreq)]
        for li in range(layers):
            pool_np = gpu_pool_to_oracle({"codes": pg.c_codes[li], "params": pg.c_params[li], "rope": pg.rope_buf[li],
                                          "hp": pg.hp_c[li], "row_of_slot": pg.hp_row_of_slot,
                                          "owner_of_row": pg.hp_owner_of_row})
            qh = st["q"][li, :nreq].float().cpu()
            ref, _ = attention.decode(pool_np, qh[..., :D], qh[..., D:], slots, lens, list(range(1, nreq + 1)), P, W,
                                      sm, D, "stored64", max_reqs=8)
            torch.testing.assert_close(og[li, :nreq].float().cpu().double(), ref, rtol=2e-2, atol=2e-3)


def test_captured_shared_decode_replays_at_other_lengths():
    """Sixteen requests that ask for more splits than there are compute units:
    the blocks are shared by what the device buffers hold at the replay. One
    captured call, replayed over equal lengths, ragged ones, requested counts that
    all fit and empty requests, back and forth, each as the same call run eagerly
    (whose scratch is its own), and against the oracle."""
    D, R, H, P, W, page, S, B, cap = 512, 64, 16, 4, 16, 64, 129, 16, 2048
    from mla_kv_quant_amd import kernels
    from tests.helpers import fused_shares, gpu_written_pool, make_queries
    assert fused_shares(B, H, D, S)
    sm = 1 / math.sqrt(192)
    gp, slots, pages, reqs = gpu_written_pool([cap] * B, D, R, P, W, page, seed=91)
    q = make_queries(B, H, D, R, sm, seed=93).to(DEV)
    pages_of = torch.from_numpy(np.stack([np.asarray(p, dtype=np.int32) for p in pages]))
    st = {"indptr": torch.zeros(B + 1, dtype=torch.int32, device=DEV),
          "indices": torch.zeros(B * cap // page, dtype=torch.int32, device=DEV),
          "seq": torch.zeros(B, dtype=torch.int64, device=DEV), "ns": torch.zeros(B, dtype=torch.int32, device=DEV),
          "req": torch.from_numpy(np.asarray(reqs)).to(DEV)}
    outs = {k: [torch.empty(B, H, S + 1, D, device=DEV), torch.empty(B, H, S + 1, device=DEV),
                torch.empty(B, H, D, dtype=torch.bfloat16, device=DEV)] for k in ("graph", "eager")}

    def set_inputs(lens, ns):
        counts = [-(-n // page) for n in lens]
        flat = torch.cat([pages_of[b, :c] for b, c in enumerate(counts)] + [torch.zeros(1, dtype=torch.int32)])
        st["indptr"].copy_(torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32))
        st["indices"][:len(flat)].copy_(flat[:st["indices"].numel()])
        st["seq"].copy_(torch.tensor(lens))
        st["ns"].copy_(torch.tensor(ns, dtype=torch.int32))

    def call(o):
        kernels.decode_fwd(q, gp["codes"], gp["params"], gp["rope"], gp["hp"], st["indptr"], st["indices"], st["seq"],
                           st["req"], st["ns"], S, o[0], o[1], o[2], sm, P, W, page, max_reqs=B + 1)

    # (the window rows in the pool are those of a sequence of `cap` tokens, so every
    # length here reads some of them at other positions: the eager call and the
    # oracle read the same ones)
    ragged = [cap, 100] + [300 + 110 * i for i in range(B - 2)]
    steps = [([1024] * B, [S] * B), (ragged, [S] * B), ([1024] * B, [S] * B), (ragged, [3 + b % 5 for b in range(B)]),
             ([0, 5, 0, cap] + [64 * i for i in range(1, B - 3)], [S] * B), ([cap] * B, [S if b % 3 else 1 for b in range(B)]),
             (ragged, [S] * B)]
    set_inputs([1] * B, [S] * B)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(outs["graph"])
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(outs["graph"])
    pool_np = gpu_pool_to_oracle(gp)
    for i, (lens, ns) in enumerate(steps):
        set_inputs(lens, ns)
        for o in outs.values():
            o[0].fill_(float("nan")), o[1].fill_(float("nan")), o[2].fill_(float("nan"))
        graph.replay()
        call(outs["eager"])
        torch.cuda.synchronize()
        og, oe = outs["graph"][2], outs["eager"][2]
        assert torch.equal(og, oe), f"replay {i} differs from the eager call"
        live = [b for b in (0, 1, 3, 7, B - 1) if lens[b]]
        ref, _ = attention.decode(pool_np, q.float().cpu()[..., :D], q.float().cpu()[..., D:], slots, lens, reqs, P, W, sm,
                                  D, "stored64", max_reqs=B + 1, batch_index=live)
        torch.testing.assert_close(og.double().cpu()[live], ref[live], rtol=2e-2, atol=2e-3)
        assert (og.cpu()[[b for b in range(B) if not lens[b]]] == 0).all()


def test_captured_extend_replays_at_other_lengths():
    """A captured extend call makes its plan on the device: replayed over other
    prefix and chunk lengths within the captured bounds it gives the bits of the
    same call run eagerly; with more key rows than it was told of, into the room
    for the plan, those of a call without that room."""
    D, R, H, P, W, page, B, T, mq, pages = 512, 64, 16, 4, 16, 16, 4, 64, 40, 600
    from mla_kv_quant_amd import kernels
    g = torch.Generator(device=DEV).manual_seed(7)
    cache = [torch.randint(0, 256, (pages * page, D // 4), dtype=torch.uint8, device=DEV, generator=g),
             torch.tensor([1.1, 1.5], device=DEV).expand(pages * page, D // 128, 2).contiguous(),
             torch.randn(pages * page, R, device=DEV, generator=g).bfloat16(),
             torch.randn(1 + (B + 1) * (P + W), D, device=DEV, generator=g).bfloat16()]
    sm = 1 / math.sqrt(192)
    q = (torch.randn(T, H, D + R, device=DEV, generator=g) * (2.0 / (sm * math.sqrt(D + R)))).bfloat16()
    kc = torch.randn(T, D + R, device=DEV, generator=g).bfloat16()
    key_rows = 9000
    spare = kernels.extend_scratch_rows(B, H, D, R, mq, key_rows)
    assert spare > 0
    st = {"qo": torch.zeros(B + 1, dtype=torch.int32, device=DEV), "indptr": torch.zeros(B + 1, dtype=torch.int32, device=DEV),
          "indices": torch.randint(0, pages, (1000,), dtype=torch.int32, device=DEV, generator=g),
          "pl": torch.zeros(B, dtype=torch.int64, device=DEV), "req": torch.arange(1, B + 1, device=DEV)}
    ws = {k: torch.empty(key_rows + spare, D + R, dtype=torch.float16, device=DEV) for k in ("graph", "eager")}
    out = {k: torch.empty(T, H, D, dtype=torch.bfloat16, device=DEV) for k in ("graph", "eager", "whole")}

    def set_inputs(prefixes, chunks):
        counts = [-(-n // page) for n in prefixes]
        st["qo"].copy_(torch.tensor(np.concatenate([[0], np.cumsum(chunks)]), dtype=torch.int32))
        st["indptr"].copy_(torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32))
        st["pl"].copy_(torch.tensor(prefixes))

    def call(o, w, rows=key_rows):
        kernels.extend_fwd(q, kc, st["qo"], st["indptr"], st["indices"], st["pl"], st["req"], *cache, mq, o, sm, P, W, page,
                           workspace=w, key_rows=rows)

    set_inputs([100] * B, [4] * B)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(out["graph"], ws["graph"])
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out["graph"], ws["graph"])
    short = ([9300, 40, 0, 0], [16, 16, 16, 16])  # 9404 key rows: into the plan's room
    steps = [([2200] * B, [16] * B), ([8000, 0, 300, 1], [40, 1, 0, 23]), ([2200] * B, [16] * B), short,
             ([0, 0, 0, 8936], [1, 20, 3, 40]), ([50] * B, [10] * B), short, ([8000, 0, 300, 1], [40, 1, 0, 23])]
    for i, (prefixes, chunks) in enumerate(steps):
        set_inputs(prefixes, chunks)
        for t in (*ws.values(), *out.values()):
            t.fill_(float("nan"))
        graph.replay()
        call(out["eager"], ws["eager"])
        rows = sum(prefixes) + sum(chunks)
        call(out["whole"], torch.empty(rows, D + R, dtype=torch.float16, device=DEV), rows)
        torch.cuda.synchronize()
        n = sum(chunks)
        assert torch.isfinite(out["whole"][:n].float()).all()
        assert torch.equal(out["graph"].view(torch.int16), out["eager"].view(torch.int16)), f"replay {i}"
        torch.testing.assert_close(out["graph"][:n].float(), out["whole"][:n].float(), rtol=2e-2, atol=2e-3)
        split = not torch.equal(out["graph"][:n], out["whole"][:n])
        assert split == (rows <= key_rows and max(prefixes) > 1000), i
