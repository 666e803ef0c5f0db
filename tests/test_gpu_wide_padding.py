"""Device binning into the wide layout when its 64-feature rows end in whole 16-feature
words without a feature (their blocks once took the negative count of features left as a
large unsigned one and read and wrote past the feature table).  Bar: exact."""
import numpy as np
import pytest

from lightgbm_rs_amd import BinMapper, HipBackend

pytestmark = pytest.mark.gpu


# feature counts with 0 to 3 empty words at a row's end, the last one in a word's middle
@pytest.mark.parametrize("F", [128, 192, 176, 161, 144, 129, 2000])
def test_empty_words_of_a_row(F):
    n = 700
    rng = np.random.default_rng(F)
    X = rng.standard_normal((F, n)).astype(np.float32)
    X[rng.random((F, n)) < 0.1] = np.nan
    ms = [BinMapper.from_column(X[f].astype(np.float64), max_bin=255) for f in range(F)]
    be = HipBackend(0)
    for col_major in (True, False):
        print(f"wide binning F={F} col_major={col_major}", flush=True)
        be.upload_raw(X if col_major else np.ascontiguousarray(X.T), ms, col_major=col_major)
        got = be.get_bins()
        for f in range(F):
            assert np.array_equal(got[f], ms[f].value_to_bin(X[f])), f
    be.close()
