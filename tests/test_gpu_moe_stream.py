"""The streamed routed-expert kernels (moe_stream.hpp): equal to the oracle, bit
for bit (exact integer sums, the same sequence of single-rounding operations),
at the edges of their row tiles, K windows and column tiles."""
import numpy as np
import pytest

from oracle import oracle
from open_rknpu2_lm_infer_amd import device as D
from open_rknpu2_lm_infer_amd import npu
from tests import refdata as R
from tests.test_gpu_ffn_moe import moe_bank, routed

pytestmark = pytest.mark.gpu


def check(h, inter, experts, dn_bits, rows, top, ids, w, tag):
    backend = npu.Backend(npu.ModelOptions(chunk=rows))
    gate, down = moe_bank(h, inter, experts, dn_bits, tag)
    moe = backend.load_moe(gate, down, top)
    x = R.activations(6, f"{tag}-x", rows, h)
    out = np.full((rows, h), np.nan, np.float32)
    print(f"{tag}: h={h} inter={inter} E={experts} W{dn_bits} rows={rows} top={top}", flush=True)
    moe.run(x, ids, w, out, rows)
    ref = oracle.moe([(g.codes, g.scales) for g in gate], [(d.codes, d.scales) for d in down], x, ids, w)
    assert np.array_equal(out, ref)


# hidden: off 16 (scalar row loads, ragged output columns), one unit, an odd
# count of W4 units, the held window's end (2048) and the reloaded one (2112 and
# 4160); intermediate: one padded unit (32), an odd count, the W8 window's end
# (1024) and past it, past the in-block quantization (2080). 65 slots and more,
# at most 10 per expert: 16-row tiles; 24 per expert: 48-row tiles or, past
# their windows, the tiled GEMM.
@pytest.mark.parametrize("dn_bits", [4, 8])
@pytest.mark.parametrize("h,inter", [(100, 32), (64, 96), (328, 160), (2048, 64), (2112, 64), (4160, 32), (128, 1024),
                                     (64, 1056), (64, 2080)])
def test_sizes(h, inter, dn_bits):
    for rows, experts in ((33, 8), (48, 4)):
        tag = f"ms-{h}-{inter}-{dn_bits}-{rows}"
        ids, w = routed(rows, experts, 2, tag)
        w[3, 1] = 0.0  # a skipped route
        check(h, inter, experts, dn_bits, rows, 2, ids, w, tag)


# Runs of exactly these lengths (0: an expert without tokens) on 16- and 48-row
# tiles, the last of a run's tiles holding one slot up to all of them.
@pytest.mark.parametrize("runs", [(1, 15, 16, 17, 0, 0, 29, 2), (64, 0, 0, 0, 0, 0, 0, 8), (15, 16, 17, 31, 32, 33),
                                  (47, 48, 49, 1, 2, 0), (90, 50, 5, 1, 0, 16, 17, 32)])
@pytest.mark.parametrize("dn_bits", [4, 8])
def test_run_lengths(runs, dn_bits):
    flat = np.repeat(np.arange(len(runs), dtype=np.int32), runs)
    R.rng_for(6, f"runs{sum(runs)}").shuffle(flat)
    rows = len(flat)
    w = R.rng_for(6, f"runs-w{rows}").uniform(0.1, 1.0, (rows, 1)).astype(np.float32)
    check(192, 96, len(runs), dn_bits, rows, 1, flat[:, None].copy(), w, f"runs-{rows}-{len(runs)}-{dn_bits}")


@pytest.mark.parametrize("h,inter,experts,dn_bits,rows,stream", [
    (64, 32, 4, 4, 72, True), (64, 32, 4, 8, 73, False),           # 36 slots per expert, both windows held
    (2112, 64, 7, 8, 35, True), (2112, 64, 7, 8, 36, False),       # 10, gate/up reloaded
    (2112, 1056, 11, 8, 33, True), (2112, 1056, 11, 8, 34, False)])  # 6, both reloaded
def test_dispatch_lines(h, inter, experts, dn_bits, rows, stream):
    """The streamed kernels up to their number of slots per expert, the tiled
    grouped GEMM past it."""
    tag = f"msd-{h}-{inter}-{rows}"
    ids, w = routed(rows, experts, 2, tag)
    with D.KernelProfile(64) as p:
        check(h, inter, experts, dn_bits, rows, 2, ids, w, tag)
    names = {s["name"] for s in p.stats if s["kind"] == 3}
    assert names == ({"moe_stream<gate_up>", "moe_stream<down>"} if stream else {"moe_gemm<gate_up>", "moe_gemm<down>"})
