"""Band modules of a plugin that provides a sweep of its own and a point
update: the sweep is the band kernel, with no kernel for whole launches
(compiled for the GPU, without one)."""
import pytest

SWEEP = r"""
#ifdef PS_BAND_COMMON
#define PS_HAS_BAND 1
template <class R>
__device__ __forceinline__ void ps_band_sweep(R *state, int gts0, int A, const ps_band_grid &g, int band, int seg)
{
    if (gts0 < 0) state[(size_t)seg * g.ny + band + A] = (R)0;
}
#endif
"""


@pytest.mark.parametrize("multi", [False, True])
def test_own_sweep_beside_a_point_update(tmp_path, monkeypatch, multi):
    from pysweep_amd import compiler, kernels
    from pysweep_amd.equations import path as eq_path
    cu = tmp_path / "both.cu"
    cu.write_text(open(eq_path("heat.cu")).read() + SWEEP)
    spec = kernels.band_spec(str(cu), 1, 1, 1, multi=multi)
    monkeypatch.setattr(compiler, "CACHE", str(tmp_path))
    code = kernels.build_module_code(spec)
    assert (b"BandMulti" if multi else b"Band") in code
    assert b"BandFull" not in code
    assert not kernels.band_has_full(spec)
    assert "full_rows" not in kernels.band_launch(spec, 64, 64)[1]
