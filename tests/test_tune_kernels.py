"""The autotuner's cache belongs to the kernels it was measured on: an entry
under another generation's key is not applied, the committed cache holds entries
of the present one only, the search starts at the engine's defaults, and chunks
of products are not searched where the factorization has none."""
import json
import os

import pytest

from mapol_amd import engine, synth, tune
from tests.test_tune import FakeEngine, clock  # noqa: F401


class LdsEngine(FakeEngine):
    def factor_form(self):
        return engine.FACTOR_LDS


def test_entry_of_other_kernels_is_not_applied(tmp_path, clock, monkeypatch):  # noqa: F811
    case, _ = synth.workload("pf118x200", T=2)
    path = str(tmp_path / "c.json")
    make = lambda **t: FakeEngine(clock, t, [])   # noqa: E731
    with monkeypatch.context() as m:
        m.setattr(tune, "KERNELS", tune.KERNELS - 1)
        old = tune.signature(case, 200, 1, 1, True)
    assert tune.tune(make, old, cache_path=path, reps=1)["cached"] is False
    new = tune.signature(case, 200, 1, 1, True)
    # the key without a generation, as caches written before it hold
    for stale in (old, new.rsplit("-k", 1)[0]):
        assert stale != new
    assert tune.tune(make, new, cache_path=path, reps=1)["cached"] is False
    assert tune.tune(make, new, cache_path=path, reps=1)["cached"] is True


def test_committed_cache_is_of_these_kernels():
    with open(tune.DEFAULT_CACHE) as fh:
        cache = json.load(fh)
    assert cache and all(k.endswith(f"-k{tune.KERNELS}") for k in cache)


def test_search_starts_at_the_defaults():
    first = {k: v[0] for k, v in {**tune.TILE_CANDIDATES, **tune.SCHEDULE_CANDIDATES}.items()}
    assert first == dict(ordering=0, tail_limit=64, chunk_products=4096, slot_chunk=1024,
                         newton_per_graph=4, tail_inverse=1, parts=1, fused_forward=1 << 20)


def test_chunk_products_only_where_there_are_chunks(tmp_path, clock):  # noqa: F811
    for kind, searched in ((FakeEngine, True), (LdsEngine, False)):
        got = tune.tune(lambda **t: kind(clock, t, []), "k", reps=1,
                        cache_path=str(tmp_path / f"{kind.__name__}.json"))
        seen = {t["tiles"]["chunk_products"] for t in got["trials"] if t["stage"] == "tiles"}
        assert (len(seen) > 1) == searched
        assert got["tiles"]["chunk_products"] == (3072 if searched else 4096)


@pytest.mark.gpu
def test_fp64_entry_runs_from_lds():
    """the tuned settings of the committed FP64 entries keep the factorization
    that the defaults run"""
    import tempfile
    import numpy as np
    from mapol_amd import matpower
    z = np.load(os.path.join(os.path.dirname(__file__), "golden", "matpower_cases.npz"))
    name = "case9241pegase"
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, name + ".m")
        matpower.write(path, float(z[f"{name}/baseMVA"]), z[f"{name}/bus"], z[f"{name}/gen"],
                       z[f"{name}/branch"])
        pegase = engine.load_matpower(path)[0]
    cache = tune.load_cache(tune.DEFAULT_CACHE)
    for case in (pegase, synth.workload("pf9241x200")[0]):
        cont = synth.n1_contingencies(case, 200, 3)
        entry = cache[tune.signature(case, 200, engine.BPF_FP64, 0, True)]
        e = engine.Engine(case, precision=engine.BPF_FP64, enforce_qlim=True, **entry["tiles"])
        tune.apply(e, entry)
        e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on)
        e.solve()
        assert e.factor_form() == engine.FACTOR_LDS
        e.close()
