"""pytest configuration: import path for the in-tree package and the `gpu` marker."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (os.path.join(ROOT, "jax-js_amd"), ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: test needs a real MI355X (run with -m gpu)")


# JAXHIP_SEED_SHIFT=<n> adds n to every integer seed the tests hand to numpy.random.default_rng: the same tests on
# other random data (shapes a test draws from its generator change with it).  Unset or 0: the committed data.
_SHIFT = int(os.environ.get("JAXHIP_SEED_SHIFT", "0"))
if _SHIFT:
    import numpy as _np

    _default_rng = _np.random.default_rng
    _np.random.default_rng = lambda seed=None: _default_rng(seed + _SHIFT if isinstance(seed, int) else seed)


# A kernel cache without kernels: the 4000 that the GPU tests compile take 11 minutes one after the other.  Processes beside the run,
# which do not see the GPU, compile those of the tests ahead of it (JAXHIP_WARM=1), each a part of them.
_warmers = []


def pytest_collection_modifyitems(items):
    part = os.environ.get("JAXHIP_WARM_PART")
    if part:
        i, n = map(int, part.split("/"))
        items[:] = [t for t in items if hasattr(t.module, "WARM_ONLY") or t.module.__name__ in ("test_parity_gpu", "test_fuzz_gpu", "test_conv")][i::n]


def pytest_collection_finish(session):
    if os.environ.get("JAXHIP_WARM") or session.config.option.collectonly or len(session.items) < 1000 or not os.path.exists("/dev/kfd"):
        return
    from jaxjs_hip.runtime import CACHE_DIR

    if os.path.isdir(CACHE_DIR) and len(os.listdir(CACHE_DIR)) > 2000:
        return
    n = max(1, int(os.environ.get("MAX_JOBS", "8")) - 4)
    for i in range(n):
        env = dict(os.environ, JAXHIP_WARM="1", JAXHIP_WARM_PART=f"{i}/{n}", HIP_VISIBLE_DEVICES="-1", OMP_NUM_THREADS="1")
        _warmers.append(subprocess.Popen([sys.executable, "-m", "pytest", os.path.join(ROOT, "tests"), "-q", "-m", "gpu", "-p", "no:cacheprovider"],
                                         cwd=ROOT, env=env, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL))


def pytest_sessionfinish():
    for p in _warmers:
        p.kill()
        p.wait()
