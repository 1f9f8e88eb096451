"""The 256x256 persistent GEMM at the edges of its pipeline: every remainder of
the scale groups in its four-group scale quads, one and several tiles per
workgroup, ragged tiles, cut tail tiles and experts of uneven size.  Each
output element takes its scale groups in order with one fp32 fma per group, as
the one-tile-per-workgroup 128x128 kernel does (held against the oracle in
test_gpu_gemm.py), so the two agree bit for bit."""
import numpy as np
import pytest
import torch

import inferop_amd
from gpu_util import device

DT = inferop_amd.dtype
TORCH_OUT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _cfg(name):
    return next(i for i in range(inferop_amd.gemm_num_configs())
                if inferop_amd.gemm_config_name(i) == name)


def _operands(m, n, k, seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    a = torch.randn((m, k), generator=g, device="cuda:0").to(torch.bfloat16)
    aq, as_ = inferop_amd.quantize(a * (1.0 + torch.arange(m, device="cuda:0")[:, None] % 7))
    bq, bs = inferop_amd.quantize_weight(torch.randn((n, k), generator=g, device="cuda:0"))
    return aq, as_, bq, bs


def _gemm(ops, m, n, k, out, name, split=1):
    c = torch.full((m, n), float("nan"), dtype=TORCH_OUT[out], device="cuda:0")
    st = inferop_amd.w8a8_block_fp8_gemm_config(c, *ops, m, n, k, getattr(DT, out), _cfg(name),
                                                split)
    assert st == 0
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (255, 129, 512), (257, 300, 768), (64, 2048, 1024),
                                   (511, 770, 1280), (4099, 4352, 256), (4096, 4610, 768),
                                   (4352, 4352, 1280)])
def test_matches_tiled_kernel(m, n, k, out):
    device()
    print(f"persist {m}x{n}x{k} {out}", flush=True)
    ops = _operands(m, n, k, m + n + k)
    want = _gemm(ops, m, n, k, out, "pre_n128_m128_w4_s2")
    assert torch.equal(_gemm(ops, m, n, k, out, "per_n256_m256_w8"), want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,split", [(300, 520, 1280, 5), (257, 2304, 1536, 2),
                                         (4096, 4608, 1792, 7)])
def test_tail_pieces(m, n, k, split):
    # a piece's sum starts from zero, so only the pieces' fp32 sums and their
    # addition differ from the whole tile's: within (split + 1) fp32 roundings
    # of the terms' magnitude, 1e-6 of the largest output here
    device()
    print(f"persist tail {m}x{n}x{k} /{split}", flush=True)
    ops = _operands(m, n, k, m + n + k)
    want = _gemm(ops, m, n, k, "fp32", "pre_n128_m128_w4_s2")
    got = _gemm(ops, m, n, k, "fp32", "per_n256_m256_w8", split)
    assert (got - want).abs().max().item() <= 1e-6 * want.abs().max().item()
    assert torch.equal(got, _gemm(ops, m, n, k, "fp32", "per_n256_m256_w8", split))


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["bf16", "fp32"])
@pytest.mark.parametrize("sizes,n,k", [([1, 0, 64, 65, 128, 129, 256, 257], 300, 768),
                                       ([3] * 33 + [0, 300], 2304, 256),
                                       ([130, 0, 0, 700], 513, 1280)])
def test_grouped_matches_per_expert(sizes, n, k, out):
    device()
    print(f"persist grouped {sizes[:4]} n={n} k={k} {out}", flush=True)
    m, e = int(sum(sizes)), len(sizes)
    aq, as_, _, _ = _operands(m, 16, k, m + n)
    bq, bs = zip(*(_operands(1, n, k, 31 * i + n)[2:] for i in range(e)))
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    c = torch.full((m, n), float("nan"), dtype=TORCH_OUT[out], device="cuda:0")
    st = inferop_amd.w8a8_block_fp8_grouped_gemm_config(
        c, aq, as_, torch.stack(bq), torch.stack(bs), torch.from_numpy(off).to("cuda:0"), m, n, k, e,
        getattr(DT, out), _cfg("per_n256_m256_w8"))
    assert st == 0
    for i in range(e):
        lo, hi = int(off[i]), int(off[i + 1])
        if hi > lo:
            want = _gemm((aq[lo:hi].contiguous(), as_[lo:hi].contiguous(), bq[i], bs[i]), hi - lo,
                         n, k, out, "pre_n128_m128_w4_s2")
            assert torch.equal(c[lo:hi], want), f"expert {i}"
