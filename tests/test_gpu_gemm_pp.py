"""The alternating-waves GEMM (large prefill tiles): every tile configuration, forced through
QLIN_GEMM_PP (a workspace reads it when it is created), against the oracle at ragged rows and
channels, at the shortest K and with several tiles per workgroup; and the rule that takes calls
to it, against the kernels it replaces (QLIN_GEMM_PP=-2), over the forms the entry points
accept.  Integer sums are exact, so plain outputs are compared bit for bit."""
import os

import numpy as np
import pytest
import torch

from open_rknpu2_lm_infer_amd import qlinear as ql
from open_rknpu2_lm_infer_amd import synth
from tests.test_gpu_parity import check_outputs, make_weights, oracle_linear

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# tile rows, weight rows, bits, plain and SiLU-gate outputs of each configuration
CONFIGS = [(256, 256, (4,), False, True), (256, 192, (4,), True, True), (256, 128, (4, 8), True, True),
           (128, 96, (4, 8), True, False), (128, 128, (4, 8), True, True), (128, 192, (4, 8), True, False),
           (128, 192, (4, 8), False, True), (128, 256, (4, 8), True, True)]


def pp_ws(cfg, rows, K, N):
    os.environ["QLIN_GEMM_PP"] = str(cfg)
    try:
        return ql.Workspace(rows, K, N)
    finally:
        del os.environ["QLIN_GEMM_PP"]


# K = 200: two k steps, fewer than the stages; K = 1152 (Kp = 1280): ten; rows one past and one
# short of a tile; channels one past a tile, and a multiple of 8 (whole-row fp16 stores)
@pytest.mark.parametrize("cfg,bits", [(c, b) for c, t in enumerate(CONFIGS) for b in t[2]])
@pytest.mark.parametrize("K,N,M", [(200, 514, 40), (1152, 390, 257), (2560, 1024, 383)])
def test_every_configuration_matches_oracle(oracle, cfg, bits, K, N, M):
    bm, bn, _, plain, swiglu = CONFIGS[cfg]
    codes = synth.codes(N, K, bits, 940 + K % 7 + bits).numpy()
    sc = synth.scales(N, bits, 941 + bits).numpy()
    w = make_weights(bits, codes, sc)
    A = synth.activations(M, K, seed=942 + M)
    R = synth.activations(M, N, seed=943)
    a, r = A.to(DEV), R.to(DEV)
    ws = pp_ws(cfg, M, K, N)
    q, s = ql.quantize(a, ldq=w.K_padded)
    if plain:
        assert ql.plan(ws, w, a)["tile_m"] == bm and ql.plan(ws, w, a)["tile_n"] == bn
        y = oracle_linear(oracle, A, codes, sc, False)
        got = ql.gemm_i32(ws, w, q)
        f32 = ql.run(ws, w, a, out_dtype=torch.float32)
        f16 = ql.run(ws, w, a, out_dtype=torch.float16)
        res = ql.run(ws, w, a, out_dtype=torch.float16, residual=r, residual_scale=0.5)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy(), oracle.gemm_i32_nk(q.cpu().numpy()[:, :K], codes))
        check_outputs(oracle, f32, y, False, torch.float32)
        check_outputs(oracle, f16, y, False, torch.float16)
        want = oracle.f32_to_f16_bits(oracle.residual_add(R.float().numpy(), y, 0.5))
        assert np.array_equal(res.cpu().view(torch.int16).numpy().view(np.uint16), want)
    if swiglu:
        assert ql.plan(ws, w, a, ql.QLIN_SWIGLU)["tile_n"] == bn // 2
        z = oracle_linear(oracle, A, codes, sc, True)
        for dt in (torch.float16, torch.float32):
            out = ql.run(ws, w, a, out_dtype=dt, flags=ql.QLIN_SWIGLU)
            torch.cuda.synchronize()
            check_outputs(oracle, out, z, True, dt)
    ws.close()
    w.close()


# several tiles per workgroup (more tiles than CUs, whole and ragged ranges per XCD), then the
# shapes around the borders of the rule
FORMS = [(4, 2560, 19456, 1100), (4, 2560, 6200, 2000), (8, 2560, 6144, 1500), (4, 4096, 2560, 1024), (8, 9728, 2560, 1100),
         (4, 1000, 5000, 777), (8, 512, 4098, 900)]


@pytest.mark.parametrize("bits,K,N,M", FORMS)
def test_rule_keeps_the_replaced_kernels_results(bits, K, N, M):
    """fp16 and f32 rows, outputs at odd strides and offsets, residuals, RMSNorm, both rounding
    modes, SiLU-gate: the same bits as the kernels that ran these before."""
    packed, _, sc = synth.make_linear(N, K, bits, 950 + M, device=DEV)
    w = ql.Weights.from_packed_device(bits, K, N, packed, sc)
    new, old = ql.Workspace(M, K, N), pp_ws(-2, M, K, N)
    A = synth.activations(M, K + 24, seed=951 + M, device=DEV, dist="student_t3")
    pl = ql.plan(new, w, A[:, :K])
    assert (pl["tile_m"], pl["waves"]) in ((256, 8), (128, 8)) and pl != ql.plan(old, w, A[:, :K]), pl
    gamma = synth.gamma(K, 952, device=DEV)
    R = synth.activations(M, N + 5, seed=953, device=DEV)
    for dt, od, pad, off in ((torch.float16, torch.float16, 0, 0), (torch.float16, torch.float16, 3, 0),
                             (torch.float32, torch.float16, 8, 1), (torch.float32, torch.float32, 0, 0),
                             (torch.float16, torch.float32, 5, 2)):
        a = A.to(dt)[:, :K] if pad else A[:, :K].to(dt).contiguous()
        for kw in (dict(), dict(flags=ql.QLIN_ROUND_HALF_EVEN, gamma=gamma), dict(residual=R.to(od)[:, off:off + N]),
                   dict(flags=ql.QLIN_SWIGLU)):
            n = N // 2 if kw.get("flags", 0) & ql.QLIN_SWIGLU else N
            got = [torch.full((M, n + pad + off), -7.0, dtype=od, device=DEV) for _ in range(2)]
            for ws, buf in zip((new, old), got):
                ql.run(ws, w, a, out=buf[:, off:off + n], **kw)
            torch.cuda.synchronize()
            assert torch.equal(*(g.view(torch.int16 if od == torch.float16 else torch.int32) for g in got)), (kw, dt, od, pad)
        # in place, as the decoder's hidden += down(...)
        got = [R.to(od)[:, :N].clone() for _ in range(2)]
        for ws, buf in zip((new, old), got):
            ql.run(ws, w, a, out=buf, residual=buf, residual_scale=0.25)
        torch.cuda.synchronize()
        assert torch.equal(*got)
    new.close()
    old.close()
    w.close()
