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
