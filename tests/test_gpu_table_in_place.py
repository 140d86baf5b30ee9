"""Location tables whose ids are written over their keys: a caller that needs
the keys no more passes one buffer for both.  The radix build allows it from
257 buckets on (its first pass has read every key before the last one writes),
so tables small enough for one launch take it too when the buffers overlap."""
import numpy as np
import pytest

from hip_mem import DeviceArray, hip
from test_gpu_location_table import closed_form

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["pt_location_table", "pt_location_table_noalloc"])
@pytest.mark.parametrize("n,K", [(1500, 257), (100_000, 545), (131_072, 8000)])
@pytest.mark.parametrize("shift", [0, 700])
def test_ids_over_the_keys(n, K, shift, entry):
    from pandemicthrust_amd.api import lib
    keys = np.random.default_rng(n + K).integers(0, K, n, dtype=np.uint32)
    print("case: %s n=%d K=%d, ids %d words behind the keys' start" % (entry, n, K, shift), flush=True)
    both = DeviceArray.from_host(np.concatenate([keys, np.zeros(shift, np.uint32)]))
    off = DeviceArray(K + 1, np.int32)
    rc = getattr(lib(), entry)(both.ptr, n, K, both.ptr.value + 4 * shift, off.ptr, 0, None)
    assert rc == 0, lib().pt_last_error()
    hip().hipDeviceSynchronize()
    want_p, want_o = closed_form(keys, K)
    assert np.array_equal(off.host(), want_o)
    assert np.array_equal(both.host().view(np.int32)[shift:shift + n], want_p)
