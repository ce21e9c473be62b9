"""GPU parity of the speech_head either side of 7 projected rows, where the
matrix cores take over from the mat-vec (head_uses_gemv,
chatterbox.cpp_amd/csrc/cbx_head.hip), against the oracle's binary64 head,
within tests/test_gpu_head.py's bound; rows of any stride, alone and in CFG
pairs."""
import numpy as np
import pytest

import oracle_lib as O
from test_gpu_head import _gpu_head, _problem, _tol, cbx, torch_cuda  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [6, 7, 9, 15])
@pytest.mark.parametrize("wtype", [O.WTYPE_F16, O.WTYPE_Q4_0, O.WTYPE_Q5_0, O.WTYPE_Q8_0])
def test_rows(cbx, torch_cuda, wtype, R):  # noqa: F811
    V, K = 331, 1024
    rng = np.random.default_rng(R + 31 * wtype)
    blocks, bias, h = _problem(rng, V, K, R, wtype)
    print(f"[gpu-case] head rows wtype={wtype} R={R}", flush=True)
    got = _gpu_head(cbx, torch_cuda, blocks, wtype, bias, h, V, K, V + 2, ld_h=K + 3)
    err = np.abs(got[:, :V].astype(np.float64) - O.head_f64(blocks, wtype, bias, h, V, K))
    assert np.all(err <= _tol(blocks, wtype, h, K)), f"{err.max():.3g}"
    assert np.all(got[:, V:] == -7.0)


@pytest.mark.parametrize("pairs", [3, 4])
def test_cfg_pairs(cbx, torch_cuda, pairs):  # noqa: F811
    torch, (mod, s) = torch_cuda, cbx
    V, K, wtype = 331, 1024, O.WTYPE_Q4_0
    rng = np.random.default_rng(pairs)
    blocks, bias, h = _problem(rng, V, K, 2 * pairs, wtype)
    d = [torch.from_numpy(x.copy()).cuda() for x in (h[:pairs], h[pairs:])]
    out = [torch.empty((pairs, V), device="cuda") for _ in range(2)]
    head = mod.Sampler.head(torch.from_numpy(np.ascontiguousarray(blocks).reshape(-1)).cuda(),
                            wtype, K, d[0], out[0], bias=torch.from_numpy(bias).cuda(),
                            hidden_uncond=d[1], logits_uncond=out[1])
    print(f"[gpu-case] head pairs={pairs}", flush=True)
    s.head_logits(head, pairs, V, V)
    torch.cuda.synchronize()
    got = np.concatenate([x.cpu().numpy() for x in out]).astype(np.float64)
    err = np.abs(got - O.head_f64(blocks, wtype, bias, h, V, K))
    assert np.all(err <= _tol(blocks, wtype, h, K)), f"{err.max():.3g}"


def _call(mod, torch, dW, wtype, db, dh, out, V, K, un=None, un_out=None):
    return mod.Sampler.head(dW, wtype, K, dh, out, bias=db, hidden_uncond=un, logits_uncond=un_out)


@pytest.mark.parametrize("R", [7, 8, 15])
@pytest.mark.parametrize("wtype", [O.WTYPE_F16, O.WTYPE_Q4_0, O.WTYPE_Q5_0, O.WTYPE_Q8_0])
def test_rows_as_in_a_larger_call(cbx, torch_cuda, wtype, R):  # noqa: F811
    """Fewer than 16 projected rows are split inside the product, 16 and more
    by a launch before it: the same rows give the same bits either way, rows
    of any stride, alone and as a CFG set, infinities and NaN staying in their
    rows.  V = 16417 gives workgroups of two row tiles to the CFG sets."""
    torch, (mod, s) = torch_cuda, cbx
    for V, K in ((331, 1024), (16417, 96)):
        rng = np.random.default_rng(R + 31 * wtype + V)
        blocks, bias, h = _problem(rng, V, K, 32, wtype)
        h[0, 5] *= 1e30
        h[1, :40] *= 1e-20
        h[2] = 0.0
        h[3, K - 1], h[4, 33] = np.inf, np.nan
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        dW, db, dh = t(blocks.reshape(-1)), t(bias), t(np.pad(h, ((0, 0), (0, 3))))
        want = torch.empty((32, V), device="cuda")
        print(f"[gpu-case] head rows wtype={wtype} R={R} V={V} beside a larger call", flush=True)
        s.head_logits(_call(mod, torch, dW, wtype, db, dh, want, V, K), 32, V, V)
        got = torch.empty((R, V), device="cuda")
        s.head_logits(_call(mod, torch, dW, wtype, db, dh[:R], got, V, K), R, V, V)
        p = min(R, 7)  # pairs: 14 projected rows at most
        c, u = torch.empty((p, V), device="cuda"), torch.empty((p, V), device="cuda")
        s.head_logits(_call(mod, torch, dW, wtype, db, dh[:p], c, V, K, dh[16:16 + p], u), p, V, V)
        torch.cuda.synchronize()
        want = want.cpu().numpy()
        same = lambda a, b: np.array_equal(a.cpu().numpy(), b, equal_nan=True)  # noqa: E731
        assert same(got, want[:R]) and same(c, want[:p]) and same(u, want[16:16 + p])
        ok = np.isfinite(h).all(1)
        assert np.isfinite(want[ok]).all() and not np.isfinite(want[~ok]).any()


def test_two_streams_of_one_handle(cbx, torch_cuda):  # noqa: F811
    """Calls of up to 15 projected rows hold nothing in the handle: two streams
    of one handle give what each call gives alone."""
    torch, (mod, s) = torch_cuda, cbx
    V, K, wtype = 6563, 1024, O.WTYPE_Q4_0
    rng = np.random.default_rng(3)
    blocks, bias, h = _problem(rng, V, K, 22, wtype)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    dW, db = t(blocks.reshape(-1)), t(bias)
    rows = [t(h[:15]), t(h[15:])]
    want = []
    for x in rows:
        o = torch.empty((len(x), V), device="cuda")
        s.head_logits(_call(mod, torch, dW, wtype, db, x, o, V, K), len(x), V, V)
        want.append(o)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[torch.zeros((len(x), V), device="cuda") for _ in range(50)] for x in rows]
    torch.cuda.synchronize()
    print("[gpu-case] head on two streams of one handle", flush=True)
    for i in range(50):
        for st, x, o in zip(streams, rows, outs):
            s.head_logits(_call(mod, torch, dW, wtype, db, x, o[i], V, K), len(x), V, V,
                          stream=st.cuda_stream)
    torch.cuda.synchronize()
    for w, o in zip(want, outs):
        assert all(torch.equal(w, x) for x in o)


def test_captured_call_outlives_a_larger_one(cbx, torch_cuda):  # noqa: F811
    """A captured call of 9 rows keeps no address that a later, larger call
    (which replaces the handle's buffer) gives back."""
    torch, (mod, s) = torch_cuda, cbx
    V, K, wtype = 700, 512, O.WTYPE_Q8_0
    rng = np.random.default_rng(4)
    blocks, bias, h = _problem(rng, V, K, 1009, wtype)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    dW, db, dh, big = t(blocks.reshape(-1)), t(bias), t(h[:9]), t(h[9:])
    want, out = torch.empty((9, V), device="cuda"), torch.zeros((9, V), device="cuda")
    head = _call(mod, torch, dW, wtype, db, dh, out, V, K)
    s.head_logits(_call(mod, torch, dW, wtype, db, dh, want, V, K), 9, V, V)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        s.head_logits(head, 9, V, V)
    many = torch.empty((1000, V), device="cuda")
    print("[gpu-case] head captured, then a larger call", flush=True)
    for n in (100, 1000):
        s.head_logits(_call(mod, torch, dW, wtype, db, big[:n], many[:n], V, K), n, V, V)
        keep = torch.full((1 << 20,), float("nan"), device="cuda")
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        del keep
