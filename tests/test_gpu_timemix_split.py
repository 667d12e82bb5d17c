"""How the time-mix prologue and epilogue share tokens and head groups out: single-wavefront workgroups below four
wavefronts per CU and workgroups of four from there, one token per wavefront and more, one head group, a partly filled
one, and many."""
import pytest

from gpu_util import say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_timemix import TOL, dev, make, ref_epilogue, ref_prologue, rel_max  # noqa: E402,F401


@pytest.mark.parametrize("M,H", [(1, 9), (127, 64), (128, 64), (129, 64), (1023, 8), (1025, 8), (8192, 1), (8193, 1),
                                 (3, 1000), (2, 9001)])
def test_split_matches_reference(dev, M, H):  # noqa: F811
    from rwkv_next_amd import kernels as K
    say("time-mix split", dict(M=M, H=H))
    t = make(dev, M, H, seed=M + H)
    ins, _ = K.timemix_prologue(t["r"], t["k"], t["v"], t["o"], t["v_first"], t["b_w"], t["b_a"], t["b_v"], t["kk_mul"],
                                t["ka_mul"], H, 64, False)
    out = K.timemix_epilogue(t["g"], t["r"], ins[2], ins[3], t["k"], t["lnx_w"], t["lnx_b"], t["r_k"], H, 64, 1e-5 * 64)
    torch.cuda.synchronize()
    for name, x, y in zip(("w", "k", "v", "a", "b"), ins[1:], ref_prologue(t, H, False)[1:]):
        assert rel_max(x, y) <= TOL, name
    assert rel_max(out, ref_epilogue(t["g"], t["r"], ins[2], ins[3], t["k"], t, H, 1e-5 * 64)) <= TOL
