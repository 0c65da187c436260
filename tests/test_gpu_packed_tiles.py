"""Per-expert kernels on the boundaries of the partial-tile packing: an expert's last row block of at most
32 / 64 rows is covered four / two column blocks to a workgroup, so every count around 32, 64 and 128 (plus a
multiple of 128) is run against every number of column blocks from one to six, where the run of column blocks
a workgroup takes ends inside, at, or beyond the matrix edge.  Same oracle and tolerances as the other
per-expert tests: bit-exact where no arithmetic precedes the quantisation."""
import pytest
import torch

from oracle import fq_oracle as O
from tests.helpers import announce, check_quant_pair, gen, randn_bf16
from tests.test_gpu_parity import EXACT, FUSED, _batched_case

pytestmark = pytest.mark.gpu

# last-block sizes on both sides of every packing boundary, alone and behind full row blocks, with empty experts
BOUNDARY_COUNTS = [1, 15, 16, 31, 32, 33, 0, 48, 63, 64, 65, 96, 127, 128, 129, 0, 128 + 31, 128 + 32, 128 + 33,
                   128 + 64, 128 + 65, 256 + 17, 256, 384 + 64, 7]


@pytest.mark.parametrize("ncb", [1, 2, 3, 4, 5, 6])
def test_batch_blockwise_quant_packing_boundaries(gpu, ncb):
    from linghe_amd.quant.block import triton_batch_blockwise_quant

    counts = BOUNDARY_COUNTS
    N = 128 * ncb
    announce("packed tiles: batch_blockwise_quant", ncb)
    x = randn_bf16(gen(70 + ncb), sum(counts), N)
    ref = O.batch_blockwise_quant(x, counts, False)
    for cdt in (torch.int32, torch.int64):
        q, s, qt, st = triton_batch_blockwise_quant(x.to(gpu), torch.tensor(counts, dtype=cdt, device=gpu), counts)
        torch.cuda.synchronize()
        check_quant_pair("packed.blockwise.row", ref[0], ref[1], q, s, **EXACT)
        check_quant_pair("packed.blockwise.col", ref[2], ref[3], qt, st, **EXACT)


@pytest.mark.parametrize("ncb", [1, 2, 3, 4, 5])
def test_batched_swiglu_packing_boundaries(gpu, ncb):
    announce("packed tiles: batched swiglu fwd/bwd", ncb)
    _batched_case(gpu, BOUNDARY_COUNTS, 256 * ncb, 1.0, 1.0, seed=80 + ncb)


@pytest.mark.parametrize("ncb", [1, 2, 3, 4, 6])
def test_pad_permute_packing_boundaries(gpu, ncb):
    """the packing goes by the PADDED row count: 17..32 real rows pad to 32 (four column blocks), 33 to 48 (two)"""
    from linghe_amd.utils.gather import triton_batch_block_pad_permute_with_indices as fn

    counts = [1, 15, 16, 17, 31, 32, 33, 0, 47, 48, 49, 63, 64, 65, 113, 128, 129, 128 + 20, 256 + 50]
    m, N = 500, 128 * ncb
    announce("packed tiles: pad+permute+quant", ncb)
    g = gen(90 + ncb)
    x = randn_bf16(g, m, N)
    probs = torch.rand(m, len(counts), generator=g)
    idx = torch.cat([torch.randperm(m, generator=g)[:c] for c in counts])
    ref = O.batch_block_pad_permute_with_indices(x, idx, probs, counts, False)
    padded = O.pad_indices(idx, counts)
    cnt = torch.tensor(counts, dtype=torch.int32, device=gpu)
    q, s, qt, st, p = fn(x.to(gpu), cnt, padded.to(gpu), counts, probs=probs.to(gpu))
    torch.cuda.synchronize()
    check_quant_pair("packed.gather.row", ref[0], ref[1], q.view(-1), s.view(-1), **EXACT)
    check_quant_pair("packed.gather.col", ref[2], ref[3], qt.view(-1), st.view(-1), **EXACT)
    assert torch.equal(p.cpu(), ref[4])


# counts for which the launch that scans them is smaller than one workgroup per tile: whole, half and quarter blocks at the
# least rows that make one (the size is then just enough), at the most, and mixed with empty experts
@pytest.mark.parametrize("counts", [[65] * 9, [33] * 9, [1] * 70, [64] * 5, [32] * 5, [65, 33, 1] * 7, [1] * 40 + [200],
                                    [0, 130, 0, 1, 2, 66, 34, 0] * 4, [300] + [3] * 90], ids=lambda c: f"{len(c)}x{c[0]}")
@pytest.mark.parametrize("ncb", [1, 3, 4, 7])
def test_scanning_launch_has_a_workgroup_for_every_tile(gpu, counts, ncb):
    from linghe_amd.quant.block import triton_batch_blockwise_quant
    from linghe_amd.utils.silu import (build_expert_plan, triton_batch_weighted_silu_and_block_quant_backward as bwd,
                                       triton_batch_weighted_silu_and_block_quant_forward as fwd)

    announce("scanning launch size", len(counts), ncb)
    x = randn_bf16(gen(ncb), sum(counts), 128 * ncb)
    ref = O.batch_blockwise_quant(x, counts, False)
    cnt = torch.tensor(counts, dtype=torch.int64, device=gpu)
    q, s, qt, st = triton_batch_blockwise_quant(x.to(gpu), cnt, counts)
    torch.cuda.synchronize()
    check_quant_pair("scan.row", ref[0], ref[1], q, s, **EXACT)
    check_quant_pair("scan.col", ref[2], ref[3], qt, st, **EXACT)
    # the SwiGLU kernels, against the launch of exactly the workgroups that have a tile
    g = gen(90 + ncb)
    h, dy = randn_bf16(g, sum(counts), 256 * ncb).to(gpu), randn_bf16(g, sum(counts), 128 * ncb).to(gpu)
    w = torch.randn(sum(counts), 1, generator=g).to(gpu)
    plan = build_expert_plan(cnt, counts)
    for fn, args in ((fwd, (h, w)), (bwd, (dy, h, w))):
        for a, b in zip(fn(*args, cnt, counts), fn(*args, cnt, counts, plan=plan)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


# column blocks that do not come in eights: every XCD takes an eighth of the tiles, column block after column block; fewer tiles
# than XCDs, eighths that end inside a column block, a last row block of the fewest rows
@pytest.mark.parametrize("M", [16, 144, 1040, 2160])
@pytest.mark.parametrize("ncb", [1, 3, 7, 9])
def test_tiles_of_shared_lines(gpu, M, ncb):
    from linghe_amd.quant.block import triton_blockwise_quant
    from linghe_amd.utils.norm import triton_rms_norm_and_block_quant_forward
    from linghe_amd.utils.silu import triton_silu_and_block_quant_forward

    announce("tiles of shared lines", M, ncb)
    n, g = 128 * ncb, gen(100 + ncb)
    x, w, h = randn_bf16(g, M, n), randn_bf16(g, n), randn_bf16(g, M, 2 * n)
    for mode in (2, 1):
        q, s, qt, st = triton_blockwise_quant(x.to(gpu), output_mode=mode)
        torch.cuda.synchronize()
        ref = O.batch_blockwise_quant(x, [M], False)
        if mode == 2:
            check_quant_pair("shared.row", ref[0], ref[1], q.view(-1), s.view(-1), **EXACT)
        check_quant_pair("shared.col", ref[2], ref[3], qt.view(-1), st.view(-1), **EXACT)
    for rows in (M, M - 1):  # transposed rows that start anywhere
        a = x[:rows].contiguous()
        q, s, rms, qt, st = triton_rms_norm_and_block_quant_forward(a.to(gpu), w.to(gpu))
        torch.cuda.synchronize()
        ref = O.rms_norm_and_block_quant_forward(a, w, rstd=rms.cpu())
        check_quant_pair("shared.rms.row", ref[0], ref[1], q, s, **EXACT)
        check_quant_pair("shared.rms.col", ref[3], ref[4], qt, st, **EXACT)
        q, s, qt, st = triton_silu_and_block_quant_forward(h[:rows].contiguous().to(gpu))
        torch.cuda.synchronize()
        ref = O.silu_and_block_quant_forward(h[:rows].contiguous())
        check_quant_pair("shared.silu.row", ref[0], ref[1], q, s, **FUSED)
        check_quant_pair("shared.silu.col", ref[2], ref[3], qt, st, **FUSED)


# the SwiGLU forward takes that order from 256 tiles on: 252, 255 and 289 of them, rows that start anywhere, and rows on half lines,
# and widths next to a multiple of 16384 columns, which stay in grid order
@pytest.mark.parametrize("M,ncb", [(2683, 12), (2160, 15), (2160, 17), (2159, 17), (2112, 17), (272, 127)])
def test_silu_tiles_of_shared_lines(gpu, M, ncb):
    from linghe_amd.utils.silu import triton_silu_and_block_quant_forward

    announce("SwiGLU tiles of shared lines", M, ncb)
    h = randn_bf16(gen(M + ncb), M, 256 * ncb)
    ref = O.silu_and_block_quant_forward(h)
    for mode in (2, 1):
        q, s, qt, st = triton_silu_and_block_quant_forward(h.to(gpu), output_mode=mode)
        torch.cuda.synchronize()
        if mode == 2:
            check_quant_pair("shared.silu.row", ref[0], ref[1], q, s, **FUSED)
        check_quant_pair("shared.silu.col", ref[2], ref[3], qt, st, **FUSED)


# RMSNorm with both outputs, rows on half lines: eighths of the tiles in grid order from 4096 columns and 3072 tiles on, 3087 of
# them here, by column blocks below, and with the transposed output alone at all sizes
@pytest.mark.parametrize("M,n", [(6208, 8064), (2112, 4224), (6208, 896)])
def test_rmsnorm_tiles_on_half_lines(gpu, M, n):
    from linghe_amd.utils.norm import triton_rms_norm_and_block_quant_forward as fn

    announce("RMSNorm tiles on half lines", M, n)
    g = gen(M + n)
    x, w = randn_bf16(g, M, n), randn_bf16(g, n)
    q, s, rms, qt, st = fn(x.to(gpu), w.to(gpu))
    qt1, st1 = fn(x.to(gpu), w.to(gpu), rms=rms, output_mode=1)[3:]
    torch.cuda.synchronize()
    ref = O.rms_norm_and_block_quant_forward(x, w, rstd=rms.cpu())
    check_quant_pair("half.rms.row", ref[0], ref[1], q, s, **EXACT)
    check_quant_pair("half.rms.col", ref[3], ref[4], qt, st, **EXACT)
    assert torch.equal(qt1.view(torch.uint8), qt.view(torch.uint8)) and torch.equal(st1, st)


# the plain quantiser takes that order from 1408 tiles on: 1404 and 1413 of them, the last row block of 112 rows; widths next to
# a multiple of 16384 columns, which stay in grid order, and one further off
@pytest.mark.parametrize("M,ncb", [(19952, 9), (20080, 9), (1424, 127), (1424, 129), (1424, 126)])
def test_plain_tiles_of_shared_lines(gpu, M, ncb):
    from linghe_amd.quant.block import triton_blockwise_quant

    announce("plain tiles of shared lines", M, ncb)
    x = randn_bf16(gen(M), M, 128 * ncb)
    ref = O.batch_blockwise_quant(x, [M], False)
    for mode in (2, 1):
        q, s, qt, st = triton_blockwise_quant(x.to(gpu), output_mode=mode)
        torch.cuda.synchronize()
        if mode == 2:
            check_quant_pair("shared.row", ref[0], ref[1], q.view(-1), s.view(-1), **EXACT)
        check_quant_pair("shared.col", ref[2], ref[3], qt.view(-1), st.view(-1), **EXACT)
