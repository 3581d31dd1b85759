"""One handle over requests of changing shapes: rotation-table rows, staging memory and captured graphs belong to the call."""
import os

import numpy as np
import pytest

from test_gpu_chunk import ckpt, ffi, make_obs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arch", ["smolvla", "pi0", "pi05"])
def test_a_handle_gives_what_a_fresh_one_gives(tmp_path, arch):
    cfg = {"smolvla": lambda: ckpt.smolvla_config(2, "bf16", suffix_mask=1), "pi0": lambda: ckpt.pi0_config(1), "pi05": lambda: ckpt.pi05_config(1)}[arch]()
    path = os.path.join(str(tmp_path), "m.vlaw")
    ckpt.write_synthetic(path, cfg, ckpt.synth_weights(cfg, seed=91))
    r = np.random.default_rng(91)
    shapes = [(2, 20, 1), (1, 5, 1), (2, 20, 1), (2, 21, 1), (3, cfg["n_lang"], 2), (1, cfg["n_lang"], 5), (2, 20, 1)]
    requests = [[make_obs(cfg, r, n_views=v, n_lang=n) for _ in range(b)] for v, n, b in shapes]
    kept = ffi.Model(path)
    for obs in requests:
        fresh = ffi.Model(path)
        for _ in range(2):  # eager, then as a captured graph
            assert np.array_equal(kept.predict_batch(obs), fresh.predict_batch(obs))
        fresh.close()
    kept.close()
