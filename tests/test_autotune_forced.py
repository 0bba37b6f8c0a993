"""Forced kernel configs (``lumen.autotune.use``, ``lumen/autotune/forced.rs``): the config classes, the
block stack, and plan cache keys that change with the forced configs."""

import pytest

import lumen_amd as L
from lumen_amd import autotune as A


def test_config_classes_and_candidates():
    gemms = A.HipGemmConfig.candidates()
    assert len(gemms) >= 5 and [c.index for c in gemms] == list(range(len(gemms)))
    with pytest.raises(ValueError):
        A.HipGemmConfig(len(gemms))
    attn = A.HipAttentionConfig.candidates()
    assert [c.waves for c in attn] == [4, 8, 2] and [c.index for c in attn] == [0, 1, 2]
    with pytest.raises(ValueError):
        A.HipAttentionConfig(waves=3)
    assert attn[0].fits(128, 128) and attn[0].fits(32, 32) and attn[0].fits(256, 256) and attn[0].fits(96, 96)
    assert attn[0].fits(64, 128) and not attn[0].fits(20, 20) and not attn[0].fits(264, 264)
    assert not attn[0].fits(64, 12)


def test_use_blocks_nest_and_key_plans():
    base = L.config.compiler.key()
    assert A.forced(A.HipGemmConfig) is None
    with A.use(A.HipGemmConfig(9)):
        assert A.forced(A.HipGemmConfig) == A.HipGemmConfig(9)
        outer = L.config.compiler.key()
        assert outer != base
        with A.use(A.HipGemmConfig(0), A.HipAttentionConfig(waves=8)):  # the inner block's config wins
            assert A.forced(A.HipGemmConfig) == A.HipGemmConfig(0)
            assert A.forced(A.HipAttentionConfig).waves == 8
            assert L.config.compiler.key() != outer
        assert A.forced(A.HipGemmConfig) == A.HipGemmConfig(9)
        assert A.forced(A.HipAttentionConfig) is None
    assert L.config.compiler.key() == base
    with pytest.raises(ValueError):
        with A.use(A.HipGemmConfig(0), A.HipGemmConfig(1)):
            pass


def test_a_flag_set_while_the_plan_key_is_worked_out_is_in_the_next_key():
    """Plan keys hold every flag as it is: one that another thread sets while a key is worked out (here: as its last
    flag is read) is in the next key, not hidden behind the kept one."""
    from lumen_amd.config import CompilerFlags

    class Raced(CompilerFlags):
        def __getattribute__(self, name):
            value = super().__getattribute__(name)
            if name == "fused_linear_cross_entropy_chunk_size" and super().__getattribute__("fuse"):
                self.fuse = False
            return value

    flags = Raced()
    flags.key()
    assert dict(flags.key())["fuse"] is False
    before = flags.key()
    assert flags.key() == before
    flags.autotune = False
    assert flags.key() != before


def test_a_forced_gemm_config_reaches_few_row_dots_with_a_consumer():
    """A dot of few rows whose consumer would run in its store is planned as a plain GEMM step inside a block that
    forces a GEMM config, which it then takes; float32 dots, which have no configs, still fuse."""
    import lumen_amd.functional as F
    from lumen_amd.compiler.plan import Plan

    def plan(dt):
        args = [L.empty(s, dt, "meta") for s in ((16, 128), (64, 128))]
        return Plan(L.make_graph(lambda x, w: F.relu(F.matmul(x, w.t(), "float32", "float32")))(*args), build_kernels=False)

    assert [st.kind for st in plan("bfloat16").steps] == ["dot"]
    with A.use(A.HipGemmConfig(0)):
        p = plan("bfloat16")
        assert [st.kind for st in p.steps] == ["dot", "loop"]
        p._apply_forced()
        assert p.steps[0].config == 0 and p.steps[0].forced
        assert [st.kind for st in plan("float32").steps] == ["dot"]
