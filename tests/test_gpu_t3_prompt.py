"""GPU parity of the prompt pass's attention tiles (t3_attn_tile,
chatterbox.cpp_amd/csrc/cbx_t3.hip) against the binary64 oracle's prompt
graph, on a small model (2 layers, n_embd 256, 4 heads of 64) so that the row
counts can take every edge: 16-row groups with one row, whole and one over,
several streams in one group, keys ending inside and at the edge of a pair of
16-key tiles, and both forms (a group per wave, or its keys split over four
waves).

Tolerance on ln_f's rows: |gpu - ref| <= 5e-5 + 5e-5 |ref|, the step tests'
(tests/test_gpu_t3.py): binary32 throughout against binary64, values O(1),
fewer layers here.
"""
import numpy as np
import pytest

import oracle_lib as O
import pkg
from oracle import cbx_t3_oracle as T3

pytestmark = pytest.mark.gpu

L_, N, H, N_POS, V = 2, 256, 4, 512, 64
TOL_ABS, TOL_REL = 5e-5, 5e-5


@pytest.fixture(scope="module")
def small():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    mod = pkg.load()
    s = mod.Sampler(device=0, max_vocab=1024, max_history=64)
    yield (torch, s) + model(torch, mod, O.WTYPE_Q8_0)
    s.close()


def model(torch, mod, wtype, N=N, H=H, sd=0.08):
    rng = np.random.default_rng(0x9A11)
    t = lambda a: torch.from_numpy(a).cuda()
    vec = lambda k, base=0.0, sd=0.1: (base + rng.standard_normal(k) * sd).astype(np.float32)
    dev, ref = [], []
    for _ in range(L_ if N == 256 else 1):
        d, r = {}, {}
        for key, o, i in (("attn_w", 3, 1), ("attn_proj_w", 1, 1), ("fc_w", 4, 1),
                          ("fc_proj_w", 1, 4)):
            # large enough that some scores stand out: the running max grows
            w = (rng.standard_normal((o * N, i * N)) * sd).astype(np.float32)
            blocks = O.quantize(w, wtype)
            d[key], r[key] = t(blocks.reshape(-1)), O.dequantize(blocks, wtype, i * N)
        for key, k, base in (("ln_1_g", N, 1.0), ("ln_1_b", N, 0.0), ("attn_b", 3 * N, 0.0),
                             ("attn_proj_b", N, 0.0), ("ln_2_g", N, 1.0), ("ln_2_b", N, 0.0),
                             ("fc_b", 4 * N, 0.0), ("fc_proj_b", N, 0.0)):
            r[key] = vec(k, base)
            d[key] = t(r[key])
        dev.append(d)
        ref.append(r)
    wpe, emb, gf, bf = vec((N_POS, N)), vec((V, N), 0.0, 0.5), vec(N, 1.0), vec(N)
    dm = mod.Sampler.t3_model(dev, t(wpe), t(emb), t(gf), t(bf), wtype=wtype, n_head=H)
    return dm, T3.Model(ref, wpe, emb, gf, bf, 1e-5, H)


def run(torch, s, dm, rows, inputs, n_slots, n_ctx, caches=None):
    """rows: (slot, position) of each input row.  Caches start as NaN (what
    was never stored must never be used) unless given."""
    if caches is None:
        k = torch.full((n_slots, L_, H, n_ctx, 64), float("nan"), device="cuda")
        caches = (k, k.clone())
    k, v = caches
    hid = torch.full((len(rows), N), 7.0, device="cuda")
    at = np.array(rows, np.int32)
    s.t3_prefill(dm, torch.from_numpy(at[:, 0].copy()).cuda(),
                 torch.from_numpy(at[:, 1].copy()).cuda(), k, v, hid,
                 inputs=torch.from_numpy(inputs).cuda())
    torch.cuda.synchronize()
    return hid.cpu().numpy(), k, v


def arranged(lens, order, rng):
    rows = [(b, p) for b, n in enumerate(lens) for p in range(n)]
    if order == "positions":   # every stream's first row, then every second ...
        rows.sort(key=lambda x: (x[1], x[0]))
    elif order == "shuffled":
        rows = [rows[i] for i in rng.permutation(len(rows))]
    return rows


CASES = [
    ((1,), "streams"), ((16,), "streams"), ((17,), "streams"), ((31,), "streams"),
    ((32,), "streams"), ((33, 1, 64, 127), "streams"), ((5, 40, 18), "positions"),
    ((70, 9, 33), "shuffled"), ((251,), "streams"),
    ((250, 129, 383) + (61,) * 60, "streams"),   # 4422 rows: a group per wave
    ((65,) * 64, "positions"),                   # 4160 rows, 16 streams in a group
]


@pytest.mark.parametrize("lens,order", CASES, ids=[f"{sum(c[0])}-{c[1]}" for c in CASES])
def test_prompt_rows_match_oracle(small, lens, order):
    """Every row and every stored key and value, some rows of each call being
    skipped ones (slot or position out of range), which give zero rows."""
    torch, s, dm, rm = small
    rng = np.random.default_rng(sum(lens) + len(order))
    rows = arranged(lens, order, rng)
    skip = set(rng.integers(0, len(rows) + 1, 3).tolist()) if len(rows) > 16 else set()
    for at in sorted(skip, reverse=True):
        rows.insert(at, [(-1, 0), (len(lens), 1), (0, 400)][at % 3])
    x = (rng.standard_normal((len(rows), N)) * 0.7).astype(np.float32)
    print(f"[gpu-case] prompt lens={lens[:4]} order={order} rows={len(rows)}", flush=True)
    got, k, v = run(torch, s, dm, rows, x, len(lens), 400)
    kr, vr = T3.new_cache(len(lens), L_, H, 400)
    where = {key: i for i, key in enumerate(rows)}
    for b, n in enumerate(lens):
        at = [where[(b, p)] for p in range(n)]
        want = T3.prefill(rm, x[at], kr, vr, b, 0)
        err = np.abs(got[at] - want)
        assert np.all(err <= TOL_ABS + TOL_REL * np.abs(want)), f"stream {b}: {err.max():.3g}"
        for c, r in ((k, kr), (v, vr)):
            c = c[b, :, :, :n].cpu().numpy()
            assert np.allclose(c, r[b, :, :, :n], rtol=TOL_REL, atol=TOL_ABS)
    good = {(b, p) for b, n in enumerate(lens) for p in range(n)}
    for i, key in enumerate(rows):
        if key not in good:
            assert np.all(got[i] == 0.0)


def test_rows_independent_of_the_rows_beside_them(small):
    """A stream's rows are bit for bit the same alone, beside others and in
    another order (both with four waves per group)."""
    torch, s, dm, _ = small
    rng = np.random.default_rng(7)
    x = {(b, p): (rng.standard_normal(N) * 0.7).astype(np.float32)
         for b in range(3) for p in range(60)}
    out = {}
    for name, rows in (("alone", [(0, p) for p in range(60)]),
                       ("beside", arranged((60, 60, 60), "streams", rng)),
                       ("shuffled", arranged((60, 60, 60), "shuffled", rng))):
        print(f"[gpu-case] independence {name}", flush=True)
        got, _, _ = run(torch, s, dm, rows, np.stack([x[r] for r in rows]), 3, 64)
        out[name] = np.stack([got[rows.index((0, p))] for p in range(60)])
    assert np.array_equal(out["alone"], out["beside"])
    assert np.array_equal(out["alone"], out["shuffled"])


@pytest.mark.parametrize("lens", [(40, 21), (70,) * 60], ids=["split-keys", "group-per-wave"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_nonfinite_row_stays_in_its_stream(small, lens, bad):
    """One prompt row that is not finite: the rows before it and the other
    streams' (in the same group) are what they are without it, bit for bit;
    the row itself and those after it are not finite."""
    torch, s, dm, _ = small
    rng = np.random.default_rng(11)
    rows = arranged(lens, "positions", rng)
    x = (rng.standard_normal((len(rows), N)) * 0.7).astype(np.float32)
    print(f"[gpu-case] nonfinite {bad} rows={len(rows)}", flush=True)
    clean, _, _ = run(torch, s, dm, rows, x, len(lens), 80)
    hit = (1, 18)
    y = x.copy()
    y[rows.index(hit), 3] = bad
    got, _, _ = run(torch, s, dm, rows, y, len(lens), 80)
    for i, (b, p) in enumerate(rows):
        if b == hit[0] and p >= hit[1]:
            assert np.isnan(got[i]).any()
        else:
            assert np.array_equal(got[i], clean[i]), (b, p)


@pytest.mark.parametrize("lens,hit", [((180, 21), (0, 140)), ((70,) * 60, (1, 50))],
                         ids=["split-keys", "group-per-wave"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_nonfinite_row_late_in_its_stream(small, lens, hit, bad):
    """The same with rows in their streams' order, so that earlier rows of the
    hit stream share its 16-row group, and the hit position past the first
    pair of key tiles that its wave takes (sums already there to add to)."""
    torch, s, dm, _ = small
    rng = np.random.default_rng(12)
    rows = arranged(lens, "streams", rng)
    at = rows.index(hit)
    assert at // 16 == (at - 2) // 16 and hit[1] >= (128 if len(rows) < 4096 else 32)
    x = (rng.standard_normal((len(rows), N)) * 0.7).astype(np.float32)
    print(f"[gpu-case] late nonfinite {bad} rows={len(rows)}", flush=True)
    clean, _, _ = run(torch, s, dm, rows, x, len(lens), 200)
    x[at, 3] = bad
    got, _, _ = run(torch, s, dm, rows, x, len(lens), 200)
    for i, (b, p) in enumerate(rows):
        if b == hit[0] and p >= hit[1]:
            assert np.isnan(got[i]).any()
        else:
            assert np.array_equal(got[i], clean[i]), (b, p)


# 672 rows is where head_mfma's c_attn takes two or four row tiles (q rows and
# the caches its outputs), 1024 rows where the products take large tiles; 8 x 1025 rows give c_attn
# and c_fc (768 and 1024 outputs) enough workgroups of 128 x 128, attn c_proj not
@pytest.mark.parametrize("wtype,lens", [
    (O.WTYPE_Q4_0, (64,) * 16), (O.WTYPE_F16, (37,) * 30), (O.WTYPE_Q5_0, (1,) * 1023 + (18,)),
    (O.WTYPE_Q8_0, (100,) * 8), (O.WTYPE_F16, (71,) * 10), (O.WTYPE_Q4_0, (75,) * 10),
    (O.WTYPE_Q8_0, (100,) * 82), (O.WTYPE_F16, (410,) * 20), (O.WTYPE_Q4_0, (391,) * 21)])
def test_many_rows_products(small, wtype, lens):
    """The products of many rows, every format, whole and partial row tiles."""
    torch, s = small[:2]
    dm, rm = model(torch, pkg.load(), wtype)
    rng = np.random.default_rng(len(lens))
    rows = arranged(lens, "streams", rng)
    x = (rng.standard_normal((len(rows), N)) * 0.7).astype(np.float32)
    print(f"[gpu-case] many rows wtype={wtype} rows={len(rows)}", flush=True)
    got, k, v = run(torch, s, dm, rows, x, len(lens), max(lens) + 1)
    at = 0
    for b, n in enumerate(lens):
        if b % 5 == 0 or b + 1 == len(lens):
            kr, vr = T3.new_cache(1, L_, H, n)
            want = T3.prefill(rm, x[at:at + n], kr, vr, 0, 0)
            err = np.abs(got[at:at + n] - want)
            assert np.all(err <= TOL_ABS + TOL_REL * np.abs(want)), f"stream {b}: {err.max():.3g}"
            for c, r in ((k, kr), (v, vr)):
                assert np.allclose(c[b, :, :, :n].cpu().numpy(), r[0, :, :, :n], rtol=TOL_REL,
                                   atol=TOL_ABS)
        at += n


@pytest.mark.parametrize("n_streams", [3, 4, 7, 15, 16, 17])
@pytest.mark.parametrize("wtype", [O.WTYPE_F16, O.WTYPE_Q4_0, O.WTYPE_Q5_0, O.WTYPE_Q8_0])
def test_step_at_the_row_edges(small, wtype, n_streams):
    """Decode steps either side of 4 streams (mat-vecs below, matrix cores from
    there) and of a whole row tile, one stream sitting the second step out."""
    torch, s = small[:2]
    dm, rm = model(torch, pkg.load(), wtype)
    rng = np.random.default_rng(100 * wtype + n_streams)
    k = torch.full((n_streams, L_, H, 8, 64), float("nan"), device="cuda")
    v = k.clone()
    pos = torch.zeros(n_streams, dtype=torch.int32, device="cuda")
    hid = torch.full((n_streams, N), 7.0, device="cuda")
    kr, vr = T3.new_cache(n_streams, L_, H, 8)
    at = np.zeros(n_streams, np.int64)
    for t in range(3):
        toks = rng.integers(0, V, n_streams).astype(np.int32)
        state = np.zeros(n_streams, np.int32)
        state[n_streams // 2] = t == 1
        print(f"[gpu-case] step wtype={wtype} streams={n_streams} t={t}", flush=True)
        s.t3_step(dm, pos, k, v, hid, tokens=torch.from_numpy(toks).cuda(),
                  state=torch.from_numpy(state).cuda())
        torch.cuda.synchronize()
        got = hid.cpu().numpy()
        want = T3.step(rm, toks, at, kr, vr, active=state == 0)
        err = np.abs(got - want)
        assert np.all(err <= TOL_ABS + TOL_REL * np.abs(want)), f"step {t}: {err.max():.3g}"
        assert np.array_equal(pos.cpu().numpy(), at)


@pytest.mark.parametrize("n_head", [4, 8, 12, 24])
def test_split_norm_widths(small, n_head):
    """The split norm where a row fills part of a wave (n_embd 256), one, one and
    a half and three waves: two steps of 5 streams, one sitting the second out,
    and 19 prompt rows."""
    torch, s = small[:2]
    dm, rm = model(torch, pkg.load(), O.WTYPE_Q8_0, 64 * n_head, n_head, sd=0.02)
    rng = np.random.default_rng(n_head)
    n = 64 * n_head
    layers = L_ if n == 256 else 1
    k = torch.full((5, layers, n_head, 24, 64), float("nan"), device="cuda")
    v = k.clone()
    kr, vr = T3.new_cache(5, layers, n_head, 24)
    x = (rng.standard_normal((19, n)) * 0.7).astype(np.float32)
    hid = torch.empty((19, n), device="cuda")
    print(f"[gpu-case] split norm n_embd={n}", flush=True)
    s.t3_prefill(dm, torch.zeros(19, dtype=torch.int32, device="cuda"),
                 torch.arange(19, dtype=torch.int32, device="cuda"), k, v, hid,
                 inputs=torch.from_numpy(x).cuda())
    torch.cuda.synchronize()
    want = T3.prefill(rm, x, kr, vr, 0, 0)
    assert np.all(np.abs(hid.cpu().numpy() - want) <= TOL_ABS + TOL_REL * np.abs(want))
    at = np.array([19, 0, 0, 0, 0], np.int64)
    pos = torch.from_numpy(at.astype(np.int32)).cuda()
    hid = torch.empty((5, n), device="cuda")
    for t in range(2):
        toks = rng.integers(0, V, 5).astype(np.int32)
        state = np.array([0, 0, t, 0, 0], np.int32)
        s.t3_step(dm, pos, k, v, hid, tokens=torch.from_numpy(toks).cuda(),
                  state=torch.from_numpy(state).cuda())
        torch.cuda.synchronize()
        want = T3.step(rm, toks, at, kr, vr, active=state == 0)
        assert np.all(np.abs(hid.cpu().numpy() - want) <= TOL_ABS + TOL_REL * np.abs(want))


GROUPED = [(1, 1), (2, 2), (3, 3), (17, 2), (64, 64), (251, 64), (1000, 7), (4096, 4096),
           (5000, 1), (5001, 4097), (14975, 64), (20000, 9000)]


@pytest.mark.parametrize("order", ["random", "runs", "interleaved"])
@pytest.mark.parametrize("n,n_slots", GROUPED, ids=[f"{n}-{b}" for n, b in GROUPED])
def test_row_groups(small, n, n_slots, order):
    """t3_group_rows (csrc/cbx_group.h): every row in one group, a group's rows
    of one slot (modulo 4096) or all skipped, in the caller's order, at most 15
    places empty per slot; nothing written past the bound."""
    import debug_t3_lib as D
    torch = small[0]
    rng = np.random.default_rng(n + n_slots)
    slots = {"random": rng.integers(0, n_slots, n), "runs": np.arange(n) * n_slots // n,
             "interleaved": np.arange(n) % n_slots}[order].astype(np.int32)
    act = (rng.random(n) < 0.9).astype(np.int32)
    slots[act == 0] = rng.choice([-5, 2 ** 31 - 1], int((act == 0).sum()))
    print(f"[gpu-case] groups {n} rows {n_slots} slots {order}", flush=True)
    got = D.groups(torch.from_numpy(act).cuda(), torch.from_numpy(slots).cuda(), n_slots)
    got = got.cpu().numpy()
    assert got.shape[0] <= min(n, n // 16 + min(n_slots, 4096) + 1)
    assert np.array_equal(np.sort(got[got >= 0]), np.arange(n)) and got.min() >= -1
    key = np.where(act != 0, slots & 4095, 4096)
    last = {}
    for g in got:
        rows = g[g >= 0]
        if rows.size == 0:
            continue
        assert np.array_equal(g[: rows.size], rows)  # the empty places last
        k = set(key[rows].tolist())
        assert len(k) == 1
        k = k.pop()
        assert k not in last or (last[k][1] == 16 and last[k][0] < rows[0])
        assert np.all(np.diff(rows) > 0)
        last[k] = (rows[-1], rows.size)


@pytest.mark.parametrize("B,L,n_slots", [(2, 30, 2), (3, 40, 3), (20, 33, 20), (300, 20, 300),
                                         (24, 9, 8200)])
def test_one_row_per_stream(small, B, L, n_slots):
    """A call of one row per stream after their prompts: the rows of a mixed
    group, each over its own stream's positions, and 2 and 3 rows (mat-vecs, keys
    and values stored by t3_kv_append) in two and three slots.  8200 slots: some
    rows of one group in slots equal modulo 4096."""
    torch, s, dm, rm = small
    rng = np.random.default_rng(B)
    at = np.arange(B) if n_slots == B else np.concatenate(
        [[b, b + 4096, b + 8192] for b in range(B // 3)])
    x = {(b, p): (rng.standard_normal(N) * 0.7).astype(np.float32)
         for b in range(B) for p in range(L)}
    print(f"[gpu-case] one row per stream B={B} L={L} slots={n_slots}", flush=True)
    first = [(b, p) for p in range(L - 1) for b in range(B)]
    last = [(b, L - 1) for b in range(B)]
    place = lambda rows: [(int(at[b]), p) for b, p in rows]
    _, k, v = run(torch, s, dm, place(first), np.stack([x[r] for r in first]), n_slots, L)
    got, _, _ = run(torch, s, dm, place(last), np.stack([x[r] for r in last]), n_slots, L, (k, v))
    for b in range(0, B, max(1, B // 24)):
        kr, vr = T3.new_cache(1, L_, H, L)
        want = T3.prefill(rm, np.stack([x[(b, p)] for p in range(L)]), kr, vr, 0, 0)[-1]
        err = np.abs(got[b] - want)
        assert np.all(err <= TOL_ABS + TOL_REL * np.abs(want)), f"stream {b}: {err.max():.3g}"


def test_captured_prompt(small):
    """A prompt call of mixed slots captured in a graph and replayed, other
    prompts run between the replays, gives the eager call's rows."""
    torch, s, dm, _ = small
    rng = np.random.default_rng(21)
    rows = arranged((30, 7, 41, 1), "positions", rng)
    at = np.array(rows, np.int32)
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    slots, pos = t(at[:, 0].copy()), t(at[:, 1].copy())
    x = t((rng.standard_normal((len(rows), N)) * 0.7).astype(np.float32))
    want, k, v = run(torch, s, dm, rows, x.cpu().numpy(), 4, 64)
    hid = torch.zeros_like(x)
    print("[gpu-case] captured prompt", flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        s.t3_prefill(dm, slots, pos, k, v, hid, inputs=x)
    for _ in range(3):
        run(torch, s, dm, rows[:50], np.ones((50, N), np.float32), 4, 64)
        k.fill_(float("nan"))
        v.fill_(float("nan"))
        hid.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(hid.cpu().numpy(), want)
