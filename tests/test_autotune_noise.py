"""The launch autotuner on a stand-in context whose kernel times are noise:
settings that no kernel of the step reads are not timed and keep the library's
defaults, and a setting that differs by noise only is not taken; one that is
faster is."""
import importlib
import types

import numpy as np
import pytest


class Context:
    """times: kernel kind -> ms from the settings in force, times noise."""

    def __init__(self, st, seed, ms):
        self.st, self.rng, self.ms = st, np.random.default_rng(seed), ms
        self.set = {"line_solver": 1, "adv_fused": 0, "adv_x_rows": 1, "nb_advect_y": 3, "nb_advect_z": 2,
                    "adv_groups_y": 0, "adv_groups_z": 4, "nb_diffuse_x": 2, "nb_diffuse_y": 8, "nb_diffuse_z": 8,
                    "x_tile": 16, "part_shape_x": 1, "part_shape_y": 1, "part_shape_z": 0, "part_bins": 0,
                    "part_max_line": 2048, "part_max_line_strided": 512, "jacobi_x": 1, "jacobi_sweeps": 12}
        self.touched = set()

    def tune(self, **kw):
        self.touched |= set(kw)
        self.set.update(kw)

    def tune_get(self, p):
        return self.set[p]

    def profile(self, on):
        pass

    def profile_read(self):
        kinds = ("advect_x", "advect_y", "advect_z", "advect_hz", "diffuse_x", "diffuse_y", "diffuse_z")
        return {k: (self.ms(k, self.set) * (1.0 + 0.03 * self.rng.standard_normal()), 2) for k in kinds}

    def step_glue(self):
        pass

    def transport_step(self, itime, use_diffusion):
        pass


def state(**kw):
    base = dict(nx=360, ny=240, nz=50, ns=15, is_periodic=False, use_cn=True)
    return types.SimpleNamespace(**{**base, **kw})


@pytest.mark.parametrize("seed", range(20))
@pytest.mark.parametrize("periodic", [False, True])
def test_settings_without_effect_keep_defaults(pkg, seed, periodic):
    at = importlib.import_module("volcano-ash3d_amd.autotune")
    T = Context(state(is_periodic=periodic), seed, lambda k, s: 1.0)
    before = dict(T.set)
    chosen = at.autotune(T, True, line_solver="partitioned")
    unread = {"nb_advect_y", "nb_advect_z", "adv_groups_y", "adv_groups_z"}
    assert not unread & (T.touched | set(chosen))
    explicit = Context(state(use_cn=False, is_periodic=periodic), seed, lambda k, s: 1.0)
    at.autotune(explicit, True)
    assert not {p for p in explicit.touched if p.startswith(("nb_diffuse", "x_tile", "part_", "jacobi"))}
    assert all(T.set[p] == before[p] for p in unread)


def test_noise_rarely_changes_a_setting(pkg):
    """3 % noise, 2 % margin, nothing faster: of 200 tunings times a dozen
    settings, few take another value (one measurement alone takes most)."""
    at = importlib.import_module("volcano-ash3d_amd.autotune")
    changed = total = 0
    for seed in range(200):
        T = Context(state(), seed, lambda k, s: 1.0)
        before = dict(T.set)
        chosen = at.autotune(T, True, line_solver="partitioned")
        total += len(chosen)
        changed += sum(v[0] != before[p] for p, v in chosen.items())
    assert changed < 0.25 * total, (changed, total)


def test_faster_settings_are_taken(pkg):
    at = importlib.import_module("volcano-ash3d_amd.autotune")
    T = Context(state(), 1, lambda k, s: 1.0 if k != "diffuse_z" or s["part_shape_z"] == 0 else 0.7)
    at.autotune(T, True, line_solver="partitioned")
    assert T.set["part_shape_z"] == 1
    T = Context(state(is_periodic=True), 1, lambda k, s: 1.0 if k != "advect_y" or s["nb_advect_y"] != 2 else 0.7)
    at.autotune(T, False)
    assert T.set["nb_advect_y"] == 2
