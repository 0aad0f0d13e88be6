"""GPU parity of the grouped MoE projection (`mxa_gemm_moe`, one launch over all experts) and of
`HipPackedMoEExperts`, the packed-GPU `QuantizedMoEExperts` (app/architectures/moe_experts.py:29-89).

Each row of the grouped launch must equal the CPU oracle's matmul of that row by its expert's
weight bit for bit. The module must equal, bit for bit, the reference's own forward loop
(moe_experts.py:81-88) run over per-expert `DevicePackedLinear`s: one call per active expert and
projection, `index_add_` in ascending expert order. Routings cover experts with no rows, an
expert with more than one 16-row chunk, a single token, all tokens on one expert, and output
widths that leave the last row tile partial.
"""

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from matricxon_amd import synthetic as S
from matricxon_amd.device_packed import DevicePackedLinear
from matricxon_amd.gemm import q8k_bytes
from matricxon_amd.moe import HipPackedMoEExperts, route_pairs
from oracle import dequant as D
from tests.test_gpu_kernels import assert_within_tolerance

pytestmark = pytest.mark.gpu

TYPES = [D.Q4_K, D.Q6_K, D.Q8_0]


def bits(a: np.ndarray) -> np.ndarray:
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def assert_bit_exact(got: np.ndarray, want: np.ndarray, what: str) -> None:
    assert got.shape == want.shape, what
    diff = np.nonzero(bits(got) != bits(want))
    assert diff[0].size == 0, (f"{what}: {diff[0].size} outputs differ, first at "
                               f"{diff[0][0]},{diff[1][0]}: {got[diff][0]} vs {want[diff][0]}")


def expert_weights(t: int, n_experts: int, n: int, k: int, seed: int) -> np.ndarray:
    """(n_experts, n, row_bytes) packed bytes, each expert its own random weight."""
    return np.stack([S.packed_weight(t, n, k, seed=seed + e) for e in range(n_experts)])


def offsets_of(counts: list[int]) -> np.ndarray:
    return np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)


# rows per expert: an empty expert first, in the middle and last; one expert past 16 rows
COUNTS = [[0, 3, 0, 37, 1, 0], [5], [1, 1, 1, 1], [0, 0, 17, 0]]


@pytest.mark.parametrize("ggml_type", TYPES)
@pytest.mark.parametrize("n,k", [(512, 1024), (300, 2048), (96, 256)])
@pytest.mark.parametrize("ci", range(len(COUNTS)))
def test_grouped_rows_match_oracle(gpu, oracle, ggml_type, n, k, ci) -> None:
    counts = COUNTS[ci]
    n_experts, n_rows = len(counts), sum(counts)
    w = expert_weights(ggml_type, n_experts, n, k, seed=n + k + ci)
    x = S.activations(n_rows, k, seed=ci + 1)
    off = offsets_of(counts)
    want = np.zeros((n_rows, n), dtype=np.float32)
    for e in range(n_experts):
        if counts[e]:
            want[off[e]:off[e + 1]] = oracle.gemm(ggml_type, w[e], x[off[e]:off[e + 1]], n, k)
    wd = torch.from_numpy(w).cuda()
    offd = torch.from_numpy(off).cuda()
    xd = torch.from_numpy(x).cuda()
    got = gpu.matmul_moe(ggml_type, wd, xd, offd, max(counts), n, k)
    assert_bit_exact(got.cpu().numpy(), want, "x quantized by the call")
    # the Q8_K activations already in the workspace (x None)
    ws = torch.empty(q8k_bytes(n_rows, k), dtype=torch.uint8, device="cuda")
    gpu.quantize_into(xd, ws)
    out = torch.full((n_rows, n), float("nan"), dtype=torch.float32, device="cuda")
    got = gpu.matmul_moe(ggml_type, wd, None, offd, max(counts), n, k, workspace=ws, out=out)
    assert_bit_exact(got.cpu().numpy(), want, "Q8_K given")


# Expert matrices of 4096 rows and more at bounds up to 32 rows, and mid-sized ones over many experts; N past
# a whole tile, an empty expert, one past 16 rows.
_MANY = [int(c) for c in np.random.default_rng(5).integers(0, 4, 40)]
GROUPED_LARGE = [(D.Q4_K, 8200, 1024, [3, 0, 5, 16, 1, 17, 2, 4]),
                 (D.Q6_K, 4100, 2048, [3, 0, 5, 16, 1, 17, 2, 4]),
                 (D.Q8_0, 8200, 512, [3, 0, 5, 16, 1, 17, 2, 4]),
                 (D.Q4_K, 4096, 1024, [2, 7, 1, 0, 9, 3, 16, 5]),
                 (D.Q4_K, 4000, 256, _MANY), (D.Q8_0, 3000, 256, _MANY), (D.Q6_K, 3000, 512, _MANY),
                 # up to 16 rows per expert
                 (D.Q6_K, 4100, 2048, [3, 0, 5, 16, 1, 12, 2, 4]),
                 (D.Q8_0, 8200, 1024, [16, 1, 0, 7, 9]),
                 (D.Q4_K, 14336, 1024, [2, 7, 1, 0, 9, 3, 16, 5]),
                 # long rows (more than 16 blocks)
                 (D.Q6_K, 4096, 14336, [3, 0, 5, 16, 1, 12, 2, 4]),
                 (D.Q4_K, 4100, 5120, [16, 2, 0, 9]), (D.Q8_0, 4096, 8192, [5, 16, 1]),
                 # several chunks of one expert
                 (D.Q6_K, 4096, 5120, [64, 0, 33, 1, 17]), (D.Q4_K, 4096, 1024, [48, 50, 3]),
                 (D.Q4_K, 4096, 1024, [90, 5, 70]), (D.Q6_K, 4096, 1024, [100, 3, 0, 40]),
                 # expert matrices of 1024 to 4096 rows
                 (D.Q4_K, 1024, 2048, [5, 0, 9, 16, 2]), (D.Q6_K, 2048, 1024, [3, 17, 1]),
                 (D.Q8_0, 1500, 4096, [7, 0, 2]), (D.Q6_K, 3072, 5120, [2, 11, 0, 4])]


@pytest.mark.parametrize("case", range(len(GROUPED_LARGE)))
def test_grouped_rows_large_experts_match_oracle(gpu, oracle, case) -> None:
    t, n, k, counts = GROUPED_LARGE[case]
    n_experts, n_rows = len(counts), sum(counts)
    w = expert_weights(t, n_experts, n, k, seed=70 + case)
    x = S.activations(n_rows, k, seed=80 + case)
    off = offsets_of(counts)
    got = gpu.matmul_moe(t, torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(),
                         torch.from_numpy(off).cuda(), max(counts), n, k).cpu().numpy()
    rows = np.unique(np.concatenate([np.arange(0, n, 37), np.arange(n - 40, n)]))
    for e in range(n_experts):
        if counts[e]:
            want = oracle.gemm(t, w[e][rows], x[off[e]:off[e + 1]], len(rows), k)
            assert_bit_exact(got[off[e]:off[e + 1]][:, rows], want, f"expert {e}")


@pytest.mark.parametrize("ggml_type", TYPES)
def test_grouped_rows_many_per_expert_match_oracle(gpu, oracle, ggml_type) -> None:
    """More than 32 rows per expert on average take 64-row chunks on the prefill tiles: experts
    with 0, 1, 63 / 64 / 65 and 150 rows (three chunks), N past a whole 128-row tile."""
    counts = [0, 150, 3, 70, 0, 64, 65, 1, 63]
    n, k = 700, 512
    n_experts, n_rows = len(counts), sum(counts)
    w = expert_weights(ggml_type, n_experts, n, k, seed=90 + ggml_type)
    x = S.activations(n_rows, k, seed=91)
    off = offsets_of(counts)
    got = gpu.matmul_moe(ggml_type, torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(),
                         torch.from_numpy(off).cuda(), max(counts), n, k).cpu().numpy()
    for e in range(n_experts):
        if counts[e]:
            want = oracle.gemm(ggml_type, w[e], x[off[e]:off[e + 1]], n, k)
            assert_bit_exact(got[off[e]:off[e + 1]], want, f"expert {e}")


# Every form of the grouped launch and every type, N past a tile, an empty expert, one past 16 rows: the
# batched-decode bodies (rows of a CU resident, in a ring, long rows), the 32-row prefill tiles (past 20 rows
# an expert on average) and, past the 256 experts that those list, two or four tile groups per workgroup
_300 = [int(c) for c in np.random.default_rng(6).integers(0, 3, 299)] + [17]
FORMS = ([(D.Q4_K, 1040, 2048, [5, 0, 17, 3]), (D.Q6_K, 1030, 4096, [5, 17, 3]),
          (D.Q8_0, 1040, 2048, [5, 0, 17, 3])] +
         [(D.Q4_K, 4100, 4096, [5, 0, 17, 3, 1, 8, 2, 4]), (D.Q6_K, 4100, 4096, [5, 0, 17, 3, 1, 8, 2, 4]),
          (D.Q8_0, 2050, 3072, [5, 0, 17, 3, 1, 2, 0, 1, 1, 1, 2, 0, 3, 1, 1, 4])] +
         [(t, 1040, 6144, [5, 0, 17]) for t in TYPES] +
         [(t, 300, 1280, [5, 31, 32, 33, 1, 40]) for t in TYPES] +
         [(D.Q4_K, 70, 512, _300), (D.Q4_K, 250, 256, _300), (D.Q6_K, 40, 512, _300), (D.Q6_K, 120, 256, _300),
          (D.Q8_0, 250, 512, _300)])


@pytest.mark.parametrize("case", range(len(FORMS)))
def test_grouped_forms_match_oracle(gpu, oracle, case) -> None:
    t, n, k, counts = FORMS[case]
    w = expert_weights(t, len(counts), n, k, seed=300 + case)
    x = S.activations(sum(counts), k, seed=330 + case)
    off = offsets_of(counts)
    bound = 16 if counts is _300 else max(counts)  # the tile's chunks loop over the last expert's 17 rows
    got = gpu.matmul_moe(t, torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(),
                         torch.from_numpy(off).cuda(), bound, n, k).cpu().numpy()
    rows = np.unique(np.concatenate([np.arange(0, n, 37), np.arange(max(0, n - 40), n)]))
    for e, c in enumerate(counts):
        if c:
            want = oracle.gemm(t, np.ascontiguousarray(w[e][rows]), x[off[e]:off[e + 1]], len(rows), k)
            assert_bit_exact(got[off[e]:off[e + 1]][:, rows], want, f"expert {e}")


def test_grouped_rows_with_loose_bound(gpu, oracle) -> None:
    """max_rows_per_expert above every expert's count (the module passes n_tokens): the extra
    16-row chunks find no rows and exit."""
    counts = [2, 0, 9]
    n, k, t = 256, 1024, D.Q4_K
    w = expert_weights(t, len(counts), n, k, seed=5)
    x = S.activations(sum(counts), k, seed=6)
    off = offsets_of(counts)
    got = gpu.matmul_moe(t, torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(),
                         torch.from_numpy(off).cuda(), 200, n, k).cpu().numpy()
    for e in range(len(counts)):
        if counts[e]:
            assert_bit_exact(got[off[e]:off[e + 1]],
                             oracle.gemm(t, w[e], x[off[e]:off[e + 1]], n, k), f"expert {e}")


# (type, N, K, bound, counts), each with experts past the bound: the decode tile (its chunks loop), the
# prefill tiles (64-row chunks, 32-row chunks) and the batched-decode bodies
PAST_BOUND = [(D.Q6_K, 256, 1024, 16, [40, 0, 3, 33]), (D.Q4_K, 300, 512, 40, [130, 0, 3, 81]),
              (D.Q6_K, 4100, 256, 16, [40, 0, 3, 33]), (D.Q8_0, 4100, 256, 20, [70, 1, 0, 45]),
              (D.Q4_K, 4096, 1024, 16, [40, 0, 3, 17]),
              (D.Q6_K, 14336, 1024, 8, [20, 5, 0, 9, 1, 16, 3, 2]),
              (D.Q8_0, 4096, 4096, 12, [16, 30, 0, 1]), (D.Q6_K, 4096, 5120, 16, [33, 2, 0, 17])]


@pytest.mark.parametrize("case", range(len(PAST_BOUND)))
def test_grouped_rows_past_the_bound(gpu, oracle, case) -> None:
    """max_rows_per_expert below an expert's count (a token routed twice to one expert gives it
    more rows than tokens): every row is still computed (the decode tile's chunks loop; the
    prefill-body forms take their (expert, chunk) list from the offsets)."""
    t, n, k, bound, counts = PAST_BOUND[case]
    w = expert_weights(t, len(counts), n, k, seed=7)
    x = S.activations(sum(counts), k, seed=8)
    off = offsets_of(counts)
    out = torch.full((sum(counts), n), float("nan"), dtype=torch.float32, device="cuda")
    got = gpu.matmul_moe(t, torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(),
                         torch.from_numpy(off).cuda(), bound, n, k, out=out).cpu().numpy()
    for e in range(len(counts)):
        if counts[e]:
            assert_bit_exact(got[off[e]:off[e + 1]],
                             oracle.gemm(t, w[e], x[off[e]:off[e + 1]], n, k), f"expert {e}")


# (n_tokens, top_k, n_experts, id dtype): decode and batched routings, more than one chunk of 1024
# pairs, more distinct experts than a wave has lanes, ids outside the range, int32 ids
ROUTE_CASES = [(1, 2, 8, torch.int64), (16, 8, 40, torch.int64), (300, 6, 256, torch.int64),
               (2000, 4, 64, torch.int32), (5, 3, 1, torch.int64), (1030, 1, 7, torch.int32),
               # one pair; a wave's run of whole steps; a last wave of one pair; runs of many steps
               (1, 1, 2, torch.int64), (512, 8, 64, torch.int64), (961, 1, 129, torch.int32),
               (9001, 4, 9, torch.int64)]


@pytest.mark.parametrize("case", range(len(ROUTE_CASES)))
def test_route_kernel_matches_route_pairs(gpu, case) -> None:
    """mxa_moe_route against the torch steps of route_pairs (a stable argsort of the clamped ids):
    the same offsets, each sorted pair's token, each pair's place and the ids as int32."""
    n_tokens, top_k, n_experts, dtype = ROUTE_CASES[case]
    g = torch.Generator().manual_seed(case)
    ids = torch.randint(-2, n_experts + 2, (n_tokens, top_k), generator=g).to(dtype).cuda()
    offsets, pair_tok, rows, ids32 = gpu.moe_route(ids, n_experts)
    order, want_off, want_tok = route_pairs(ids, n_experts)
    assert torch.equal(offsets.cpu(), want_off.cpu())
    assert torch.equal(pair_tok.cpu().long(), want_tok.cpu())
    want_rows = torch.empty_like(order)
    want_rows[order] = torch.arange(order.numel(), device=order.device)
    assert torch.equal(rows.cpu().long().reshape(-1), want_rows.cpu())
    assert torch.equal(ids32.cpu(), ids.cpu().to(torch.int32))


def test_route_pairs_on_device_matches_host() -> None:
    idx = torch.tensor([[3, 0], [1, 3], [0, 2], [3, 1]], device="cuda")
    order, offsets, pair_tok = route_pairs(idx, 5)
    assert offsets.cpu().tolist() == [0, 2, 4, 5, 8, 8]
    assert order.cpu().tolist() == [1, 4, 2, 7, 5, 0, 3, 6]
    assert pair_tok.cpu().tolist() == [0, 2, 1, 3, 2, 0, 1, 3]


def reference_forward(x, top_k_weights, top_k_idx, per_expert, activation):
    """The reference's QuantizedMoEExperts.forward (moe_experts.py:81-88) over per-expert
    DevicePackedLinear modules: gate, up, down per active expert in ascending id order."""
    n_tokens, n_embd = x.shape
    out = torch.zeros(n_tokens, n_embd, dtype=torch.float32, device=x.device)
    for expert_id in top_k_idx.unique().tolist():
        gate_m, up_m, down_m = per_expert[expert_id]
        token_idx, k_idx = (top_k_idx == expert_id).nonzero(as_tuple=True)
        x_e = x.index_select(0, token_idx)
        gate = activation(gate_m(x_e.unsqueeze(0)).squeeze(0))
        up = up_m(x_e.unsqueeze(0)).squeeze(0)
        down = down_m((gate * up).unsqueeze(0)).squeeze(0)
        weight = top_k_weights[token_idx, k_idx].unsqueeze(-1)
        out.index_add_(0, token_idx, (down * weight).to(torch.float32))
    return out.to(x.dtype)


def build_experts(types, n_experts, n_embd, ffn_len, dtype, seed):
    gt, ut, dt = types
    gate = expert_weights(gt, n_experts, ffn_len, n_embd, seed)
    up = expert_weights(ut, n_experts, ffn_len, n_embd, seed + 100)
    down = expert_weights(dt, n_experts, n_embd, ffn_len, seed + 200)
    mod = HipPackedMoEExperts.from_packed_bytes(gate.tobytes(), up.tobytes(), down.tobytes(),
                                                types, n_experts, n_embd, ffn_len, F.silu, dtype,
                                                torch.device("cuda"))
    per_expert = [tuple(DevicePackedLinear(torch.from_numpy(np.ascontiguousarray(w[e])).cuda(),
                                           k, t, None, dtype)
                        for w, k, t in ((gate, n_embd, gt), (up, n_embd, ut), (down, ffn_len, dt)))
                  for e in range(n_experts)]
    return mod, per_expert


def routing(n_tokens, n_experts, top_k, seed, device="cuda"):
    g = torch.Generator().manual_seed(seed)
    logits = torch.randn(n_tokens, n_experts, generator=g)
    w, idx = torch.topk(torch.softmax(logits, dim=-1), top_k, dim=-1)
    return (w / w.sum(-1, keepdim=True)).to(device), idx.to(device)


MODULE_CASES = [
    # (types gate/up/down, n_experts, n_embd, ffn_len, n_tokens, top_k, dtype)
    ((D.Q4_K, D.Q4_K, D.Q6_K), 8, 1024, 512, 24, 2, torch.float32),
    # one token on the pairs launch (every projection's K / 256 in the kernel's set)
    ((D.Q4_K, D.Q4_K, D.Q6_K), 8, 4096, 2048, 1, 2, torch.bfloat16),
    ((D.Q8_0, D.Q8_0, D.Q4_K), 16, 2048, 2048, 1, 4, torch.float32),
    ((D.Q8_0, D.Q8_0, D.Q8_0), 4, 512, 768, 7, 2, torch.float32),
    ((D.Q4_K, D.Q4_K, D.Q4_K), 16, 512, 256, 40, 4, torch.bfloat16),
    ((D.Q6_K, D.Q6_K, D.Q4_K), 8, 256, 512, 1, 2, torch.float32),
    # one bfloat16 token through the fused steps, the down projection on 56-block rows
    ((D.Q4_K, D.Q4_K, D.Q6_K), 4, 1024, 14336, 1, 2, torch.bfloat16),
    # experts of 1024 rows and more: OLMoE-like 64 experts top 8, long down rows, float32 and Q8_0 down
    ((D.Q4_K, D.Q4_K, D.Q6_K), 64, 2048, 1024, 16, 8, torch.bfloat16),
    ((D.Q4_K, D.Q4_K, D.Q6_K), 64, 2048, 1024, 64, 8, torch.bfloat16),
    ((D.Q4_K, D.Q4_K, D.Q6_K), 8, 1024, 5120, 12, 2, torch.bfloat16),
    ((D.Q6_K, D.Q6_K, D.Q8_0), 6, 2048, 1024, 20, 2, torch.float32),
]


@pytest.mark.parametrize("case", range(len(MODULE_CASES)))
def test_module_matches_reference_loop(case) -> None:
    types, n_experts, n_embd, ffn_len, n_tokens, top_k, dtype = MODULE_CASES[case]
    mod, per_expert = build_experts(types, n_experts, n_embd, ffn_len, dtype, seed=case * 7)
    x = torch.from_numpy(S.activations(n_tokens, n_embd, seed=case + 3)).cuda().to(dtype)
    tw, tidx = routing(n_tokens, n_experts, top_k, seed=case)
    got = mod(x, tw, tidx)
    want = reference_forward(x, tw, tidx, per_expert, F.silu)
    assert got.dtype == want.dtype == dtype
    assert torch.equal(got.float().view(torch.int32), want.float().view(torch.int32)), \
        f"max |diff| {(got.float() - want.float()).abs().max().item()}"


def test_module_all_tokens_on_one_expert() -> None:
    types = (D.Q4_K, D.Q4_K, D.Q4_K)
    mod, per_expert = build_experts(types, 4, 256, 256, torch.float32, seed=11)
    n_tokens = 33  # three 16-row chunks for the one expert
    x = torch.from_numpy(S.activations(n_tokens, 256, seed=12)).cuda()
    tidx = torch.full((n_tokens, 1), 2, dtype=torch.int64, device="cuda")
    tw = torch.rand(n_tokens, 1, generator=torch.Generator().manual_seed(1)).cuda()
    got = mod(x, tw, tidx)
    want = reference_forward(x, tw, tidx, per_expert, F.silu)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_module_repeated_expert_in_a_tokens_routing(dtype) -> None:
    """Every token names expert 2 in both slots (and a few name expert 1 twice): expert 2 gets
    2 * n_tokens rows, more than the launch is sized for; the reference computes both slots."""
    types = (D.Q4_K, D.Q4_K, D.Q6_K)
    n_tokens = 20
    mod, per_expert = build_experts(types, 4, 512, 256, dtype, seed=31)
    _check_repeated_routing(mod, per_expert, n_tokens, 512)


@pytest.mark.parametrize("n_tokens,ffn", [(40, 256), (20, 4096)])
def test_module_repeated_expert_past_the_bound_on_prefill_tiles(n_tokens, ffn) -> None:
    """The same repeated routing at a bound past 32 rows and with a 4096-row expert matrix."""
    types = (D.Q4_K, D.Q4_K, D.Q6_K)
    mod, per_expert = build_experts(types, 4, 512, ffn, torch.bfloat16, seed=34)
    _check_repeated_routing(mod, per_expert, n_tokens, 512)


def _check_repeated_routing(mod, per_expert, n_tokens: int, n_embd: int) -> None:
    x = torch.from_numpy(S.activations(n_tokens, n_embd, seed=32)).cuda().to(mod.dtype)
    tidx = torch.full((n_tokens, 2), 2, dtype=torch.int64, device="cuda")
    tidx[::7] = 1
    tw = torch.rand(n_tokens, 2, generator=torch.Generator().manual_seed(33)).cuda()
    got = mod(x, tw, tidx)
    want = reference_forward(x, tw, tidx, per_expert, F.silu)
    assert torch.equal(got.float().view(torch.int32), want.float().view(torch.int32)), \
        f"max |diff| {(got.float() - want.float()).abs().max().item()}"


def test_module_rejects_types_without_a_kernel() -> None:
    z = torch.zeros((2, 256, 144), dtype=torch.uint8, device="cuda")
    with pytest.raises(ValueError):  # Q5_K (13): no HIP kernel
        HipPackedMoEExperts(z, z, z, 13, 13, 13, 256, 256, F.silu)


# the grouped launch's forms: the decode tile, the prefill tiles (64-row chunks, 32-row ones over 40
# experts) and, for IQ4_XS, the float-row kernel
GROUPED_BF16 = [(D.Q4_K, 512, 1024, COUNTS[0]), (D.Q6_K, 300, 2048, COUNTS[0]),
                (D.Q8_0, 700, 512, [0, 150, 3, 70, 0, 64, 65, 1, 63]),
                (D.Q4_K, 700, 512, [0, 150, 3, 70, 0, 64, 65, 1, 63]),
                (D.Q4_K, 4000, 256, _MANY), (D.IQ4_XS, 512, 1024, COUNTS[0])]


@pytest.mark.parametrize("case", range(len(GROUPED_BF16)))
def test_grouped_bf16_equal_the_float32_result_cast(gpu, case) -> None:
    """`mxa_gemm_moe_bf16` writes each output as the float32 launch's value rounded by torch's
    cast, bit for bit, on float rows and on prequantized Q8_K blocks (x None)."""
    t, n, k, counts = GROUPED_BF16[case]
    n_experts, n_rows = len(counts), sum(counts)
    w = torch.from_numpy(expert_weights(t, n_experts, n, k, seed=200 + case)).cuda()
    x = torch.from_numpy(S.activations(n_rows, k, seed=210 + case)).cuda()
    off = torch.from_numpy(offsets_of(counts)).cuda()
    want = gpu.matmul_moe(t, w, x, off, max(counts), n, k)
    got = gpu.matmul_moe(t, w, x, off, max(counts), n, k, out_dtype=torch.bfloat16)
    assert got.dtype == torch.bfloat16 and got.shape == want.shape
    assert torch.equal(got.view(torch.int16), want.to(torch.bfloat16).view(torch.int16))
    if t != D.IQ4_XS:
        ws = torch.empty(q8k_bytes(n_rows, k), dtype=torch.uint8, device="cuda")
        gpu.quantize_into(x, ws)
        pre = gpu.matmul_moe(t, w, None, off, max(counts), n, k, workspace=ws,
                             out=torch.empty((n_rows, n), dtype=torch.bfloat16, device="cuda"),
                             out_dtype=torch.bfloat16)
        assert torch.equal(pre.view(torch.int16), got.view(torch.int16))


@pytest.mark.parametrize("n,k", [(512, 1024), (300, 2048)])
@pytest.mark.parametrize("ci", range(len(COUNTS)))
def test_grouped_iq4_xs_rows_equal_single_rows(gpu, n, k, ci) -> None:
    """IQ4_XS experts in the grouped launch (float activations): every row equals mxa_gemm of
    that row alone bit for bit, and an expert's rows equal mxa_gemm of them together while the
    expert has up to 16 (from 17 rows mxa_gemm takes the matrix cores: within tolerance)."""
    counts = COUNTS[ci]
    n_experts, n_rows = len(counts), sum(counts)
    w = expert_weights(D.IQ4_XS, n_experts, n, k, seed=n + k + ci)
    x = S.activations(n_rows, k, seed=ci + 11)
    off = offsets_of(counts)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    got = gpu.matmul_moe(D.IQ4_XS, wd, xd, torch.from_numpy(off).cuda(), max(counts), n, k)
    got = got.cpu().numpy()
    for e in range(n_experts):
        for r in range(off[e], off[e + 1]):
            alone = gpu.matmul(D.IQ4_XS, wd[e], xd[r:r + 1], n, k).cpu().numpy()
            assert_bit_exact(got[r:r + 1], alone, f"expert {e} row {r}")
        if counts[e]:
            together = gpu.matmul(D.IQ4_XS, wd[e], xd[off[e]:off[e + 1]], n, k).cpu().numpy()
            if counts[e] <= 16:
                assert_bit_exact(got[off[e]:off[e + 1]], together, f"expert {e}")
            else:
                assert_within_tolerance(got[off[e]:off[e + 1]], together)


# up to 16 tokens an expert has at most 16 rows (top-k ids are distinct): bit for bit, also in
# bfloat16; 24 float32 tokens may give an expert 17+ rows
@pytest.mark.parametrize("n_tokens,dtype", [(1, torch.bfloat16), (10, torch.bfloat16),
                                            (6, torch.float32), (24, torch.float32)])
def test_module_iq4_xs_experts_match_reference_loop(n_tokens, dtype) -> None:
    """An IQ4_XS expert set (gate/up IQ4_XS, down Q4_K) in the grouped launch, with no host sync:
    bit for bit the reference's loop while every expert has up to 16 rows, within tolerance of it
    otherwise (an expert with 17+ rows in the loop runs mxa_gemm's matrix-core prefill)."""
    types = (D.IQ4_XS, D.IQ4_XS, D.Q4_K)
    mod, per_expert = build_experts(types, 4, 1024, 512, dtype, seed=41 + n_tokens)
    assert not mod._pairs
    x = torch.from_numpy(S.activations(n_tokens, 1024, seed=42)).cuda().to(dtype)
    tw, tidx = routing(n_tokens, 4, 2, seed=43)
    got = mod(x, tw, tidx)
    want = reference_forward(x, tw, tidx, per_expert, F.silu)
    assert got.dtype == want.dtype == dtype
    rows_per_expert = torch.bincount(tidx.reshape(-1).cpu(), minlength=4)
    if int(rows_per_expert.max()) <= 16:
        assert torch.equal(got.float().view(torch.int32), want.float().view(torch.int32))
    else:
        assert_within_tolerance(got.float().cpu().numpy(), want.float().cpu().numpy())


PAIR_CASES = [
    # (type, n_experts, out, in, n_pairs, x shared by the pairs)
    (D.Q4_K, 8, 1024, 4096, 2, True),
    (D.Q4_K, 8, 1000, 4096, 8, False),
    (D.Q6_K, 4, 512, 2048, 3, True),
    (D.Q8_0, 6, 777, 2048, 4, False),
    (D.Q6_K, 3, 256, 14336, 2, False),  # 56-block rows: x quantized into the workspace first
    (D.Q4_K, 2, 4096, 14336, 1, True),
    (D.Q4_K, 4, 20000, 4096, 2, True),  # row sets: more rows than one pass holds
]


@pytest.mark.parametrize("case", range(len(PAIR_CASES)))
def test_pairs_rows_match_oracle(gpu, oracle, case) -> None:
    t, n_experts, n, k, n_pairs, shared = PAIR_CASES[case]
    w = expert_weights(t, n_experts, n, k, seed=case * 11)
    ids = np.random.default_rng(case).permutation(n_experts)[:n_pairs].astype(np.int32)
    x = S.activations(1 if shared else n_pairs, k, seed=case + 5)
    got = gpu.matmul_moe_pairs(t, torch.from_numpy(w).cuda(), torch.from_numpy(ids).cuda(),
                               torch.from_numpy(x).cuda(), n, k)
    assert got is not None, "the pairs launch declined a shape it is built for"
    got = got.cpu().numpy()
    for p in range(n_pairs):
        xr = x[:1] if shared else x[p:p + 1]
        assert_bit_exact(got[p:p + 1], oracle.gemm(t, w[ids[p]], xr, n, k), f"pair {p}")


@pytest.mark.parametrize("case", range(len(PAIR_CASES)))
def test_pairs_bf16_equal_the_float32_result_cast(gpu, case) -> None:
    """The bfloat16 pairs launch (bfloat16 x read in the kernel, bfloat16 y) equals the float32
    launch on the bfloat16 values of x, cast by torch; on Q8_K blocks (x None) it equals it too."""
    t, n_experts, n, k, n_pairs, shared = PAIR_CASES[case]
    w = torch.from_numpy(expert_weights(t, n_experts, n, k, seed=case * 13)).cuda()
    ids = torch.from_numpy(np.random.default_rng(case + 50).permutation(n_experts)[:n_pairs]
                           .astype(np.int32)).cuda()
    xb = torch.from_numpy(S.activations(1 if shared else n_pairs, k, seed=case + 9)).cuda().to(torch.bfloat16)
    want = gpu.matmul_moe_pairs(t, w, ids, xb.float(), n, k)
    got = gpu.matmul_moe_pairs(t, w, ids, xb, n, k, out_dtype=torch.bfloat16)
    assert got is not None and got.dtype == torch.bfloat16
    assert torch.equal(got.view(torch.int16), want.to(torch.bfloat16).view(torch.int16))
    ws = torch.empty(q8k_bytes(xb.shape[0], k), dtype=torch.uint8, device="cuda")
    gpu.quantize_into(xb.float(), ws)
    pre = gpu.matmul_moe_pairs(t, w, ids, None, n, k, workspace=ws, x_rows=xb.shape[0],
                               out_dtype=torch.bfloat16)
    assert torch.equal(pre.view(torch.int16), got.view(torch.int16))


def test_pairs_decline_shapes_they_do_not_take(gpu) -> None:
    ids = torch.zeros(1, dtype=torch.int32, device="cuda")
    w = torch.zeros((2, 64, 3 * 144), dtype=torch.uint8, device="cuda")  # K = 768: 3 blocks
    x = torch.zeros((1, 768), dtype=torch.float32, device="cuda")
    assert gpu.matmul_moe_pairs(D.Q4_K, w, ids, x, 64, 768) is None
    w = torch.zeros((2, 64, 4 * 210), dtype=torch.uint8, device="cuda")  # rows of 840 bytes
    x = torch.zeros((1, 1024), dtype=torch.float32, device="cuda")
    assert gpu.matmul_moe_pairs(D.Q6_K, w, ids, x, 64, 1024) is None


def combine_reference(down, rows, ids, weights, bf16):
    """The module's torch combine restated on the CPU: per token, slots in stable ascending id
    order, `down.to(dtype)` (bf16: rounded) times the float32 weight added to a float32 zero."""
    n_tokens, top_k = ids.shape
    out = torch.zeros(n_tokens, down.shape[1], dtype=torch.float32)
    for t in range(n_tokens):
        for k in torch.argsort(ids[t], stable=True).tolist():
            v = down[rows[t, k]]
            if bf16:
                v = v.to(torch.bfloat16).to(torch.float32)
            out[t] = out[t] + v * weights[t, k]
    return out


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("n_tokens,top_k,n_embd", [(1, 2, 4096), (5, 8, 1000), (3, 16, 300)])
def test_moe_combine_matches_torch_steps(gpu, bf16, n_tokens, top_k, n_embd) -> None:
    # repeated expert ids (slot order decides), rows in a shuffled order, and special values: NaN,
    # infinities, -0.0 and float32 values halfway between two bfloat16 values (ties to even)
    g = torch.Generator().manual_seed(n_tokens * 100 + top_k + int(bf16))
    total = n_tokens * top_k
    down = torch.randn(total, n_embd, generator=g) * 8
    down[0, :6] = torch.tensor([float("nan"), float("inf"), -0.0, 1 + 2 ** -8, 1 + 3 * 2 ** -8,
                                -float("inf")])
    ids = torch.randint(0, max(2, top_k // 2), (n_tokens, top_k), generator=g, dtype=torch.int32)
    rows = torch.randperm(total, generator=g).to(torch.int32).view(n_tokens, top_k)
    weights = torch.rand(n_tokens, top_k, generator=g)
    weights[0, 0] = -0.0
    got = gpu.moe_combine(down.cuda(), ids.cuda(), weights.cuda(), rows.cuda(), round_bf16=bf16)
    want = combine_reference(down, rows, ids, weights, bf16)
    got = got.cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    fin = ~torch.isnan(want)
    assert torch.equal(got[fin].view(torch.int32), want[fin].view(torch.int32))
    # identity rows (NULL): pair p's row is p
    got2 = gpu.moe_combine(down.cuda(), ids.cuda(), weights.cuda(), None, round_bf16=bf16).cpu()
    ident = torch.arange(total, dtype=torch.int32).view(n_tokens, top_k)
    want2 = combine_reference(down, ident, ids, weights, bf16)
    fin2 = ~torch.isnan(want2)
    assert torch.equal(torch.isnan(got2), torch.isnan(want2))
    assert torch.equal(got2[fin2].view(torch.int32), want2[fin2].view(torch.int32))


def test_module_bf16_routing_weights_take_the_torch_combine() -> None:
    # routing weights in bfloat16: the product stays bfloat16 in torch, so the module keeps the
    # torch combine; still the reference loop's bits
    types = (D.Q4_K, D.Q4_K, D.Q6_K)
    mod, per_expert = build_experts(types, 8, 4096, 2048, torch.bfloat16, seed=21)
    x = torch.from_numpy(S.activations(1, 4096, seed=22)).cuda().to(torch.bfloat16)
    tw, tidx = routing(1, 8, 2, seed=23)
    tw = tw.to(torch.bfloat16)
    got = mod(x, tw, tidx)
    want = reference_forward(x, tw, tidx, per_expert, F.silu)
    assert torch.equal(got.float().view(torch.int32), want.float().view(torch.int32))
