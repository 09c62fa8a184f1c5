"""The eigensolver's work space never shrinks as the batch grows: callers size it
for their largest batch and run a shorter last one in the same space."""

import pytest

import calcir_amd as C

# both sides of every line between the routes
SIZES = [1, 65, 66, 128, 129, 192, 193, 256, 257, 511, 512, 1023, 1024, 1025, 2048, 2079, 2080, 2081, 3104, 3105, 5000]


@pytest.mark.parametrize("prec", [C.PREC_FP32, C.PREC_BF16X3, C.PREC_FP64], ids=["fp32", "bf16x3", "fp64"])
@pytest.mark.parametrize("det", ["0", "1"])
@pytest.mark.parametrize("stages", [None, "1", "2"])
def test_workspace_grows_with_the_batch(prec, det, stages, monkeypatch):
    monkeypatch.setenv("CIR_DETERMINISTIC", det)
    if stages:
        monkeypatch.setenv("CIR_EIGH_STAGES", stages)
    ws = C.lib().cir_eigh_workspace
    for n in SIZES:
        ld = (n + 3) // 4 * 4
        last = 0
        for batch in list(range(1, 70)) + [127, 128, 200, 201, 256, 511, 512]:
            got = ws(prec, batch, n, ld)
            assert got >= last, (n, batch, got, last)
            last = got
