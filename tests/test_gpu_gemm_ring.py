"""GPU parity of the NF4 GEMM's ring kernel (``nf4_gemm_k2``: bf16, K % 128 == 0, r <=
16, blocksize >= 64): the edges of its tiles (64, 128, 256 rows and columns), of its
superstages (one, two and odd numbers of 128 K values, whose second K group is empty or
shorter), ranks that are no multiple of 8, and each tile and form (plain, K split, SiLU).

Tolerances of the other NF4 GEMM tests: 1e-2 of the largest output, and 98 % of the
outputs bit-identical to the oracle (only the float32 summation order differs).
"""

import ctypes

import numpy as np
import pytest
import torch

from conftest import rel_err, to_dev_bf16
from oracle.bf16 import bf16_bits_to_f32
from test_gemm_plan import plan
from test_gpu_gemm import _check
from test_gpu_nf4 import _code, make_linear_case, oracle_linear, run_linear

pytestmark = pytest.mark.gpu

# m, n, k, r, bias, blocksize, (rows, columns, K groups, K slices)
CASES = [
    (65, 72, 128, 16, True, 64, (64, 64, 2, 1)),     # one superstage: the second K group has none
    (66, 80, 384, 5, True, 128, (64, 64, 2, 1)),     # 2 + 1, r % 8 != 0 (scalar LoRA B loads)
    (129, 1027, 640, 1, False, 64, (64, 64, 2, 1)),  # 3 + 2, N % 8 != 0 (element stores), rank 1
    (513, 320, 256, 0, True, 256, (64, 64, 2, 1)),   # an absmax block of two superstages
    (257, 4104, 896, 12, True, 64, (64, 128, 2, 1)), # 4 + 3
    (257, 3600, 1920, 0, True, 64, (64, 128, 2, 1)),
    (1030, 2056, 128, 16, True, 64, (128, 128, 1, 1)),   # several rounds of workgroups
    (1025, 16392, 256, 0, True, 64, (128, 128, 1, 1)),
    (200, 8208, 640, 16, True, 64, (128, 128, 2, 1)),
    (200, 8208, 896, 0, False, 64, (128, 128, 2, 1)),
    (2049, 4104, 512, 0, True, 64, (256, 256, 1, 1)),  # one row and 8 columns past the tiles
    # K split, each tile that has it with and without LoRA
    (200, 528, 1920, 16, True, 64, (64, 64, 2, 4)),
    (140, 96, 4224, 0, False, 64, (64, 64, 2, 9)),
    (65, 2064, 4224, 16, True, 64, (64, 128, 2, 6)),
    (65, 2320, 7936, 0, True, 64, (64, 128, 2, 6)),
    (65, 3600, 4224, 0, True, 64, (128, 128, 1, 7)),
    (65, 6192, 3456, 16, True, 64, (128, 128, 1, 9)),
    (65, 4112, 4224, 0, False, 64, (128, 128, 2, 6)),
    (65, 4112, 4224, 16, True, 64, (128, 128, 2, 6)),
]


@pytest.mark.parametrize("m,n,k,r,with_bias,bs,tile", CASES)
def test_ring_gemm_matches_oracle(dev, m, n, k, r, with_bias, bs, tile):
    assert plan(m, n, k, r, bs) == tile  # what the case is for
    print(f"ring gemm m={m} n={n} k={k} r={r} bias={with_bias} bs={bs}", flush=True)
    c = make_linear_case(m + n + k + r, m, n, k, r, with_bias, bs=bs)
    _check(run_linear(dev, c), oracle_linear(c))


def test_ring_gemm_without_a_workspace_runs_unsplit(dev):
    """The K split needs its workspace; without one the same call runs unsplit and
    agrees with the oracle too."""
    from grpo_mi355x import _lib

    lib = _lib.device_library()
    m, n, k, r = 140, 96, 4224, 16
    assert lib.grpo_nf4_lora_linear_workspace_bytes(m, n, k, r, 1, 64) > 0
    c = make_linear_case(7, m, n, k, r, True)
    x, bias, a, b = (to_dev_bf16(c[key], dev) for key in ("x", "bias", "a", "b"))
    packed, absmax = (torch.from_numpy(c[key]).to(dev) for key in ("packed", "absmax"))
    y = torch.empty((m, n), dtype=torch.bfloat16, device=dev)
    arr, seg = ctypes.c_void_p * 4, (ctypes.c_int * 4)(n, 0, 0, 0)
    _lib.check(lib.grpo_nf4_lora_linear_grouped(
        x.data_ptr(), k, packed.data_ptr(), absmax.data_ptr(), _code(dev).data_ptr(), 64, 1, seg,
        arr(bias.data_ptr()), arr(a.data_ptr()), arr(b.data_ptr()), r, 2.0, y.data_ptr(), n, m, k,
        None, 0, _lib.stream_handle(dev)), "grpo_nf4_lora_linear_grouped")
    torch.cuda.synchronize()
    _check(y.view(torch.int16).cpu().numpy().view(np.uint16), oracle_linear(c))


def test_ring_gemm_infinite_t_reaches_only_its_ranks(dev):
    """A rank whose x . A overflows gives inf * B, as the reference's sum over the r
    ranks does, and no NaN from the tile's unused ranks (inf * 0)."""
    m, n, k, r = 70, 64, 256, 3
    c = make_linear_case(9, m, n, k, r, False)
    big = np.full(k, 0x7F7F, np.uint16)  # the largest bf16
    c["a"] = c["a"].copy()
    c["a"][2] = big
    c["x"] = c["x"] & np.uint16(0x7FFF)  # non-negative: t overflows to +inf
    c["b"] = np.abs(bf16_bits_to_f32(c["b"])).astype(np.float32).view(np.uint32)
    c["b"] = ((c["b"] >> 16).astype(np.uint16) | np.uint16(0x3C00)) & np.uint16(0x3FFF)
    y = bf16_bits_to_f32(run_linear(dev, c))
    assert np.all(np.isposinf(y))


@pytest.mark.parametrize("m,i,k,tile", [
    (65, 8, 128, (128, 128, 1, 1)), (130, 1000, 384, (128, 128, 1, 1)),
    (1030, 264, 896, (128, 128, 2, 1)), (513, 17416, 256, (128, 128, 1, 1)),
    (513, 8200, 384, (256, 256, 1, 1))])  # one row and 8 columns past the tiles
def test_ring_gate_up_silu_matches_float32(dev, m, i, k, tile):
    """SiLU(gate) * up of the stacked weight against the same formula on the oracle's
    bf16 gate and up: two roundings after them, so 2^-7 of the largest output."""
    from grpo_mi355x import _lib

    assert plan(m, i, k, 0, silu=1) == tile
    lib = _lib.device_library()
    c = make_linear_case(m + i + k, m, 2 * i, k, 0, False)
    gu = torch.from_numpy(bf16_bits_to_f32(oracle_linear(c)))
    g, u = gu[:, :i], gu[:, i:]
    ref = ((g * torch.sigmoid(g)).bfloat16().float() * u).bfloat16().float().numpy()
    x = to_dev_bf16(c["x"], dev)
    packed, absmax = (torch.from_numpy(c[key]).to(dev) for key in ("packed", "absmax"))
    for pad in (8, 3):  # 16-byte and element stores
        act = torch.zeros((m, i + pad), dtype=torch.bfloat16, device=dev)
        _lib.check(lib.grpo_nf4_gate_up_silu(
            x.data_ptr(), k, packed.data_ptr(), absmax.data_ptr(), _code(dev).data_ptr(), 64, i,
            k, m, act.data_ptr(), i + pad, _lib.stream_handle(dev)), "grpo_nf4_gate_up_silu")
        torch.cuda.synchronize()
        assert torch.all(act[:, i:] == 0)
        got = act[:, :i].float().cpu().numpy()
        assert np.all(np.isfinite(got)) and rel_err(got, ref) <= 2.0 ** -7
