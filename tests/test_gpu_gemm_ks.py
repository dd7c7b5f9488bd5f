"""The wave-split-K GEMM (a few to a few hundred quantized rows): every tile configuration,
forced through QLIN_GEMM_KS (a workspace reads it when it is created), against the oracle at
ragged rows and channels and at K steps that do not divide among the waves; and the rule that
takes calls to it, against the kernels it replaces (QLIN_GEMM_KS=-2), over the forms the entry
points accept.  Integer sums are exact, so plain outputs are compared bit for bit."""
import os

import numpy as np
import pytest
import torch

from open_rknpu2_lm_infer_amd import qlinear as ql
from open_rknpu2_lm_infer_amd import synth
from tests.test_gpu_parity import check_outputs, make_weights, oracle_linear

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
CONFIGS = 20


def ks_ws(cfg, rows, K, N):
    os.environ["QLIN_GEMM_KS"] = str(cfg)
    try:
        return ql.Workspace(rows, K, N)
    finally:
        del os.environ["QLIN_GEMM_KS"]


# K = 200: two k steps, fewer than the waves; K = 1152: nine; M and N: one row and channel past
# a tile, one short of it, and several tiles of the smallest configuration
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("K,N,M", [(200, 50, 9), (1152, 98, 97), (2560, 194, 33)])
def test_every_configuration_matches_oracle(oracle, bits, K, N, M):
    codes = synth.codes(N, K, bits, 900 + K % 7 + bits).numpy()
    sc = synth.scales(N, bits, 901 + bits).numpy()
    w = make_weights(bits, codes, sc)
    A = synth.activations(M, K, seed=902 + M)
    R = synth.activations(M, N, seed=903)
    a, r = A.to(DEV), R.to(DEV)
    y, z = oracle_linear(oracle, A, codes, sc, False), oracle_linear(oracle, A, codes, sc, True)
    q, s = ql.quantize(a, ldq=w.K_padded)
    acc = oracle.gemm_i32_nk(q.cpu().numpy()[:, :K], codes)
    seen = set()
    for cfg in range(CONFIGS):
        ws = ks_ws(cfg, M, K, N)
        pl = ql.plan(ws, w, a, ql.QLIN_NO_FUSED_QUANT)
        seen.add((pl["tile_m"], pl["tile_n"], pl["waves"]))
        got = ql.gemm_i32(ws, w, q)
        out = ql.run(ws, w, a, out_dtype=torch.float32, flags=ql.QLIN_NO_FUSED_QUANT)
        res = ql.run(ws, w, a, out_dtype=torch.float16, flags=ql.QLIN_NO_FUSED_QUANT, residual=r, residual_scale=0.5)
        act = ql.run(ws, w, a, out_dtype=torch.float16, flags=ql.QLIN_NO_FUSED_QUANT | ql.QLIN_SWIGLU)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy(), acc), cfg
        check_outputs(oracle, out, y, False, torch.float32)
        want = oracle.f32_to_f16_bits(oracle.residual_add(R.float().numpy(), y, 0.5))
        assert np.array_equal(res.cpu().view(torch.int16).numpy().view(np.uint16), want), cfg
        check_outputs(oracle, act, z, True, torch.float16)
        ws.close()
    # every configuration of W4, and of W8 those whose rings fit the LDS
    assert len(seen) >= CONFIGS - (0 if bits == 4 else 3), seen
    w.close()


FORMS = [(bits, K, N, M) for bits in (4, 8) for K, N, M in
         ((2560, 6144, 9), (2560, 6144, 24), (2560, 2000, 65), (4096, 2560, 100), (9728, 2560, 33), (1000, 999, 200),
          (2560, 19456, 24), (4096, 2560, 300), (256, 17, 128))]


@pytest.mark.parametrize("bits,K,N,M", FORMS)
def test_rule_keeps_the_replaced_kernels_results(bits, K, N, M):
    """fp16 and f32 rows, row strides beyond K and N, outputs and residuals at odd strides and
    offsets, RMSNorm, both rounding modes, SiLU-gate for even N: the same bits as before."""
    packed, _, sc = synth.make_linear(N, K, bits, 910 + M, device=DEV)
    w = ql.Weights.from_packed_device(bits, K, N, packed, sc)
    new, old = ql.Workspace(M, K, N), ks_ws(-2, M, K, N)
    A = synth.activations(M, K + 24, seed=911 + M, device=DEV, dist="student_t3")
    assert ql.plan(new, w, A[:, :K], ql.QLIN_NO_FUSED_QUANT)["tile_m"] in range(16, 97)
    gamma = synth.gamma(K, 912, device=DEV)
    for dt in (torch.float16, torch.float32):
        for a in (A[:, :K].to(dt).contiguous(), A.to(dt)[:, :K], A.to(dt)[:, 3:K + 3]):
            for pad, off in ((0, 0), (3, 0), (8, 1)):
                for od in (torch.float16, torch.float32):
                    forms = [dict(), dict(flags=ql.QLIN_ROUND_HALF_EVEN), dict(gamma=gamma)]
                    forms.append(dict(residual=synth.activations(M, N + 5, seed=913, device=DEV).to(od)[:, off:off + N],
                                      residual_scale=1.5))
                    if N % 2 == 0:
                        forms.append(dict(flags=ql.QLIN_SWIGLU))
                    for kw in forms:
                        kw["flags"] = kw.get("flags", 0) | ql.QLIN_NO_FUSED_QUANT
                        n = N // 2 if kw["flags"] & ql.QLIN_SWIGLU else N
                        got = [torch.full((M, n + pad + off), -7.0, dtype=od, device=DEV) for _ in range(2)]
                        for ws, buf in zip((new, old), got):
                            ql.run(ws, w, a, out=buf[:, off:off + n], **kw)
                        torch.cuda.synchronize()
                        assert torch.equal(*(g.view(torch.int16 if od == torch.float16 else torch.int32) for g in got)), kw
    new.close()
    old.close()
    w.close()


def test_rule_takes_one_round_of_workgroups():
    """Where no configuration covers the output in one round of workgroups, the kernels stay."""
    K, N = 2560, 19456
    packed, _, sc = synth.make_linear(N, K, 4, 920, device=DEV)
    w = ql.Weights.from_packed_device(4, K, N, packed, sc)
    ws = ql.Workspace(512, K, N)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for M in (9, 16, 17, 32, 33, 64, 128, 256, 512):
        pl = ql.plan(ws, w, synth.activations(M, K, seed=921, device=DEV), ql.QLIN_NO_FUSED_QUANT)
        if 0 < pl["tile_m"] <= 96:
            assert pl["grid"] <= cus and pl["grid"] == -(-M // pl["tile_m"]) * -(-N // pl["tile_n"]), pl
        else:
            assert M > 64, (M, pl)
    ws.close()
    w.close()


def test_search_keeps_the_planners_kernel(tmp_path):
    """A variant search whose candidates are all slower than the planner's kernel leaves that
    in use, in the table and after its file is read back."""
    ql.tune_clear()
    K, N, M = 4096, 2560, 64
    packed, _, sc = synth.make_linear(N, K, 4, 930, device=DEV)
    w = ql.Weights.from_packed_device(4, K, N, packed, sc)
    ws = ql.Workspace(M, K, N)
    A = synth.activations(M, K, seed=931, device=DEV)
    before, out = ql.plan(ws, w, A), ql.run(ws, w, A)
    ql.tune(ws, w, M, reps=5)
    assert ql.tune_count() == 1 and ql.plan(ws, w, A) == before
    f = tmp_path / "t.txt"
    ql.tune_save(str(f))
    ql.tune_clear()
    assert ql.tune_load(str(f)) == 1 and ql.plan(ws, w, A) == before
    again = ql.run(ws, w, A)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    ql.tune_clear()
    ws.close()
    w.close()


# shapes at which an estimate once took a slow kernel: few k steps under large tiles, few k steps into
# many channels, W8 tiles of 96 channels and a number of tiles not a multiple of 8 over a long K, many
# rows over a long K, a few rows of a wide SiLU-gate over a long K
@pytest.mark.parametrize("bits,K,N,M,swiglu", [(4, 512, 7680, 167, False), (8, 512, 2176, 512, False),
                                               (4, 66, 20000, 35, False), (8, 8576, 2944, 219, True),
                                               (8, 6400, 384, 2728, False), (4, 6016, 384, 2836, False),
                                               (4, 10000, 6252, 7, True)])
def test_choice_and_the_kernels_left_out_agree(bits, K, N, M, swiglu):
    """The chosen kernel, the kernels without these two, and a configuration of each: the same bits."""
    packed, _, sc = synth.make_linear(N, K, bits, 990 + M, device=DEV)
    w = ql.Weights.from_packed_device(bits, K, N, packed, sc)
    a = synth.activations(M, K, 991).to(DEV)
    flags = ql.QLIN_NO_FUSED_QUANT | (ql.QLIN_SWIGLU if swiglu else 0)
    got, plans = [], []
    for env in ({}, {"QLIN_GEMM_KS": "-2", "QLIN_GEMM_PP": "-2"}, {"QLIN_GEMM_KS": "10"}, {"QLIN_GEMM_PP": "2"}):
        os.environ.update(env)
        try:
            ws = ql.Workspace(M, K, N)
        finally:
            for k in env:
                del os.environ[k]
        plans.append(ql.plan(ws, w, a, flags=flags))
        got.append(ql.run(ws, w, a, out_dtype=torch.float16, flags=flags).cpu())
        ws.close()
    assert len({tuple(sorted(p.items())) for p in plans}) >= 3, plans
    assert all(torch.equal(g.view(torch.int16), got[0].view(torch.int16)) for g in got[1:])
    w.close()
