"""Prompts through fl_prefill (GEMM passes over many tokens) against the oracle's batched forward:
the cache rows that it writes and the logits of the step after it, at the edges of its tiles (64 and
128 tokens), of its attention's blocks of 64 and 128 rows, key parts and passes of 1024 tokens."""
import pytest
import torch

from tests.helpers import check_rows, fill_kv_random, log, make_pair, oracle_pair

pytestmark = pytest.mark.gpu


def _check(name, eng, orc, n, pos, seed, chunk=32):
    from flint_amd.generate import prefill
    args = eng.config
    if pos:
        fill_kv_random(eng, orc, pos, seed=seed)
    toks = torch.randint(0, args.vocab_size, (n + 1,), generator=torch.Generator().manual_seed(seed), dtype=torch.int32)
    nxt = prefill(eng, toks[:n].to(eng.device), pos, chunk=chunk)
    lg = torch.empty(args.vocab_size, dtype=torch.float32, device=eng.device)
    eng.decode_step(toks[n:].to(eng.device), pos + n, logits=lg)
    eng.check()

    def run():
        out = orc.forward(toks, pos)[0].float()
        return out, orc.k_cache[:, :, pos:pos + n].clone().float(), orc.v_cache[:, :, pos:pos + n].clone().float()

    (alt, ak, av), (ref, rk, rv) = oracle_pair(orc, run)
    for nm, got, a, r in (("k", eng.k_cache, ak, rk), ("v", eng.v_cache, av, rv)):
        got = got[:, :, pos:pos + n].cpu().float()
        # layer 0's rows: one linear of the same inputs, so only fp32 order (one rounding in a few
        # hundred, by an ulp); later layers: as far as the oracle's own implementations are apart
        e0 = float((got[0] - r[0]).norm() / r[0].norm())
        e, f = float((got - r).norm() / r.norm()), float((a - r).norm() / r.norm())
        log(f"{name} prompt {n} at {pos}: {nm} rows layer 0 rel {e0:.2e}, all {e:.2e} (oracle's two: {f:.2e})")
        assert e0 <= 2.0 ** -8 / 4 and e <= max(2 * f, 2.0 ** -8)
    check_rows(lg.cpu().view(1, -1), ref[n:], alt[n:], name, f"{name} prompt {n} at {pos}")
    # the token that prefill returns is the argmax of its last row, or ties with it
    row, am = ref[n - 1], int(nxt.item())
    assert float(row.max() - row[am]) <= 2.0 * float((alt[n - 1] - row).abs().max()) + 2.0 ** -5


@pytest.mark.parametrize("n,pos", [(17, 40), (33, 0), (63, 5), (64, 0), (65, 300), (127, 1), (129, 0), (333, 250), (700, 100)])
def test_prefill_small(dev, n, pos):
    args, sd, eng, orc = make_pair("small", seed=3)
    eng.setup_caches(1, 1100)
    orc.setup_caches(eng.max_seq_length)
    _check("small", eng, orc, n, pos, seed=n)


@pytest.mark.parametrize("chunk", [16, 31, "no memory"])
def test_prefill_verify_launches(dev, chunk, monkeypatch):
    """A prompt over several verify launches, the last one partial: with a chunk below 32, and with the default
    one where memory has no room for fl_prefill's workspace."""
    args, sd, eng, orc = make_pair("small", seed=3)
    eng.setup_caches(1, 128)
    orc.setup_caches(eng.max_seq_length)
    asked = []

    def refuse(*a):
        asked.append(a)
        raise torch.OutOfMemoryError("no room")

    monkeypatch.setattr(eng, "prefill", refuse)
    _check("small", eng, orc, 70, 5, seed=71, chunk=32 if chunk == "no memory" else chunk)
    assert len(asked) == (chunk == "no memory")


@pytest.mark.parametrize("name,n,pos", [("tiny", 1000, 0), ("tiny", 40, 900), ("tiny", 20, 1000), ("flint-3b-l1", 100, 2000),
                                        ("wide", 90, 7), ("42 heads", 840, 2100), ("flint-3b-l1", 600, 0)])
def test_prefill_shapes(dev, name, n, pos):
    """Few KV heads; a short prompt behind many keys (key parts); the 3B layer; the widest rows; enough
    rows for the large GEMM tiles (2688 weight rows: the last tile is half empty) and, behind enough
    keys, for the attention's one-way form; 320 large tiles, where gate/up takes smaller ones."""
    over = {}
    if name == "42 heads":
        name, over = "flint-3b-l1", dict(n_head=42, n_local_heads=3, dim=2688, vocab_size=2048)
    args, sd, eng, orc = make_pair(name, seed=4, weight_device="cuda", **over)
    eng.setup_caches(1, n + pos + 1)
    orc.setup_caches(eng.max_seq_length)
    _check(name, eng, orc, n, pos, seed=n)


def test_prefill_passes_and_errors(dev):
    """More tokens than one pass; the last slots of the cache, and past them; a bad token id."""
    from flint_amd import _lib
    from flint_amd.generate import prefill
    args, sd, eng, orc = make_pair("tiny", seed=5, block_size=2048)
    eng.setup_caches(1, 1100)
    toks = torch.randint(0, args.vocab_size, (1100,), generator=torch.Generator().manual_seed(6), dtype=torch.int32).to(dev)
    prefill(eng, toks, 0)
    k = eng.k_cache.clone()
    prefill(eng, toks[:1024], 0)  # the same rows in two calls
    prefill(eng, toks[1024:], 1024)
    eng.check()
    assert torch.equal(eng.k_cache, k)
    with pytest.raises(_lib.FlError) as e:
        prefill(eng, toks[:1000], eng.max_seq_length - 999)
    assert e.value.code == -2
    bad = toks[:40].clone()
    bad[7] = args.vocab_size
    prefill(eng, bad, 0)
    with pytest.raises(_lib.FlError) as e:
        eng.check()
    assert e.value.code == -1
    eng.reset_state()
    eng.check()


def test_prefill_graph_replay(dev):
    """Captured into a HIP graph, a prompt replays to the eager result (replayed several times with
    eager work between)."""
    args, sd, eng, orc = make_pair("tiny", seed=7)
    eng.setup_caches(1, 256)
    toks = torch.randint(0, args.vocab_size, (200,), generator=torch.Generator().manual_seed(8), dtype=torch.int32).to(dev)
    out = torch.empty(1, dtype=torch.int32, device=dev)
    eng.prefill(toks, 0, out)
    torch.cuda.synchronize()
    want, k, v = int(out.item()), eng.k_cache.clone(), eng.v_cache.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        eng.prefill(toks, 0, out)
    for _ in range(4):
        eng.k_cache.zero_()
        eng.v_cache.zero_()
        out.fill_(-1)
        eng.prefill(toks.flip(0).contiguous(), 0, torch.empty_like(out))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert int(out.item()) == want and torch.equal(eng.k_cache, k) and torch.equal(eng.v_cache, v)
