"""The tuner keeps the library's own shapes and plans where nothing else is faster (GPU)."""
import pytest

from pgj import _lib, tune
from pgj.mixed import MixedResident

pytestmark = pytest.mark.gpu


def test_tuner_times_the_default():
    """A tuned FP32 set: the library's choice is among the candidates, and what was recorded is the fastest."""
    print('tuner with defaults 48^3', flush=True)
    m = MixedResident(48)
    try:
        choice = m.tune(reps=2)
        for k in ('fxy', 'fz', 'fxyi'):
            ms = choice['fft'][k]['ms']
            best = min(ms, key=ms.get)
            assert choice['fft'][k]['plan'] == (int(best) if ms[best] <= tune.MARGIN * ms['0'] else 0)
        assert tune.fft_plans(m.op.grid, 4) == tuple(choice['fft'][k]['plan'] for k in ('fxy', 'fz', 'fxyi'))
        out = (_lib.c_int * 5)()
        _lib.check(_lib.lib().pgj_hex8_get_shape(m.op.grid, 6, 4, out))
        assert choice['row_march']['shape'] == tuple(out)[:4]
    finally:
        tune.reset(m.op.grid, 6, 4)
