"""Which kernel forms the coarse cross term: the pools of the resident-columns comparison (tests/test_gpu_pq_cols.py) do run
with 96 and 64 columns in LDS, a pool below four blocks a CU and the full pose term run in tiles, tables that do not pair
by rotations, FP32 on its own kernel.  If the rule moves, the comparison's sizes have to move with it."""
import pytest

from rome_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,coarse,n,order,mode,kernel,columns",
                         [("fp16", 16, 1250, 2, "list", "paired_columns", 96), ("bf16", 18, 1251, 2, "list", "paired_columns", 96),
                          ("fp16", 32, 1280, 2, "list", "paired_columns", 64), ("fp16", 16, 1250, 2, "full", "paired", 0),
                          ("fp16", 16, 300, 2, "list", "paired", 0), ("bf16", 16, 8, 1, "list", "rotations", 0),
                          ("fp32", 16, 8, 1, "list", "fp32", 0)])
def test_kernel(engine, precision, coarse, n, order, mode, kernel, columns):
    print(f"[cross term form {precision} coarse={coarse} n={n} {mode}]", flush=True)
    prob, batch, _ = synth.make_problem(is3d=True, ori=32, current=32, coarse=coarse, K=1, order=order, offset_range=5.0,
                                        n=n, snr=0.5, seed=3)
    synth.load_engine(engine, prob, precision=precision)
    try:
        engine.set_coarse_mode(mode)
        engine.reset_sums()
        engine.expectation(batch)
        assert engine.cross_term() == {"kernel": kernel, "columns": columns}
    finally:
        engine.set_coarse_mode("list")
