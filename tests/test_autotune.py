"""The batch tuner's choices on a context whose timings are made up: the launch
rule (0) is a candidate and stays unless a fixed shape is clearly faster, waves
are timed where the forward kernel reads them, and entries of other kernels are
not found."""
import pytest

import jax_cosmo_amd as jc
from jax_cosmo_amd import autotune


class FakeContext:
    def __init__(self, ms, forward_options=(1, 0)):
        self.ms, self.forward_options = ms, list(forward_options)
        self.tiles, self.variant, self.calls = (0, 0), 0, []

    def tracer_set(self, entries):
        return 1

    def get_tiles(self):
        return self.tiles

    def set_tiles(self, w, c):
        self.tiles = (w, c)

    def set_tables_variant(self, v):
        self.variant = v

    def profile(self, on):
        pass

    def angular_cl(self, *a):
        self.calls.append(self.tiles + (self.variant,))

    def profile_read(self):
        ms = self.ms(*self.tiles, self.variant)
        return {k: (v, 1) for k, v in zip(("tables", "wl", "limber"), ms)}


PROBES = [jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, 0.8)])]


@pytest.fixture(autouse=True)
def cache(tmp_path, monkeypatch):
    monkeypatch.setenv("JAX_COSMO_AMD_TUNE_CACHE", str(tmp_path / "tiles.json"))
    monkeypatch.setattr(autotune, "_device_name", lambda: "gfx")


def test_the_rule_stays_where_it_is_as_fast():
    ctx = FakeContext(lambda w, c, v: (1.0 - 0.01 * v, 1.0 - 0.002 * c, 1.0))
    best = autotune.tune_batch(PROBES, 40, n_ell=100, ctx=ctx)
    assert (best["waves"], best["wl_ctile"], best["tables_variant"]) == (0, 0, 0)
    assert {c[0] for c in ctx.calls} == {0}  # the table kernel has its own waves
    assert {c[1] for c in ctx.calls} == {0, 1, 4, 8, 16}
    autotune.apply_batch(ctx, 40, 100, 512, 1)
    assert (ctx.tiles, ctx.variant) == ((0, 0), 0)


def test_a_faster_shape_is_taken():
    ctx = FakeContext(lambda w, c, v: (1.0 - 0.2 * (v == 2), 1.0 - 0.5 * (c == 8), 1.0 - 0.5 * (w == 4)))
    for n_ell, options, waves in ((100, (1, 0), 0), (63, (1, 0), 4), (100, (0, 0), 4), (100, (1, 1), 4)):
        ctx.forward_options = list(options)
        best = autotune.tune_batch(PROBES, 40, n_ell=n_ell, ctx=ctx)
        assert (best["waves"], best["wl_ctile"], best["tables_variant"]) == (waves, 8, 2)
        autotune.apply_batch(ctx, 40, n_ell, 512, 1)
        assert (ctx.tiles, ctx.variant) == ((waves, 8), 2)


def test_entries_of_other_kernels_are_not_found():
    autotune._store({"gfx|batch|B64|L100|N512|T1": {"waves": 4, "wl_ctile": 1},
                     "gfx|server|N256|C8": {"waves": 4, "wl_ctile": 1}})
    assert autotune.lookup_batch(40, 100, 512, 1) is None
    assert autotune.lookup_server((256,), 8) is None
