"""An autotuner cache of this GPU that was measured with another version of the solver is not used."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tuned(nk, tmp_path_factory):
    path = tmp_path_factory.mktemp("tune") / "tune.txt"
    cross, _ = nk.Context(0).tune(str(path))
    return path.read_text().replace("crossover %d\n" % cross, "crossover 320\n")


@pytest.mark.parametrize("solver", [None, "", "solver 0", "solver 1000000"])
def test_cache_of_another_solver_is_ignored(nk, tuned, tmp_path, monkeypatch, solver):
    lines = tuned.splitlines()
    if solver is not None:
        lines = [solver if ln.startswith("solver ") else ln for ln in lines if solver or not ln.startswith("solver ")]
    path = tmp_path / "tune.txt"
    path.write_text("\n".join(lines) + "\n")
    monkeypatch.setenv("NRGK_TUNE_CACHE", str(path))
    assert nk.Context(0).crossover() == ((320, True) if solver is None else (768, False))
