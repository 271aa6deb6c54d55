"""What the built kernels take of the register file: the occupancies their
launch rules count on, and no spills where every loop turn would pay for them
(no GPU; the built library's own metadata)."""
import os

import pytest

from sde_mc_amd import build
from tests import kernel_notes

if not os.path.exists(build.lib_path()):
    pytest.skip('library not built', allow_module_level=True)

KERNELS = kernel_notes.kernels()


@pytest.mark.parametrize('cls,waves', [(0, 7), (1, 6), (2, 7), (3, 7), (4, 7), (5, 5), (6, 7),
                                       (7, 7), (8, 7)])
def test_batched_class_kernels_do_not_spill(cls, waves):
    for unroll in (1, 2):
        k = KERNELS.get('k_batch<%d, %d>' % (cls, unroll))
        assert k is not None or (unroll == 2 and cls not in (0, 4, 8))
        if k is None:
            continue
        assert k.get('.vgpr_spill_count', 0) == 0 and k['.private_segment_fixed_size'] == 0
        assert kernel_notes.waves_per_simd(k) >= waves


def test_control_variate_kernels_keep_their_wavefronts():
    # the 1-D Merton kernel's workgroups of eight rest on four wavefronts per SIMD
    assert kernel_notes.waves_per_simd(KERNELS['k_cv_adapted<1, 0, false>']) >= 4
    for name, k in KERNELS.items():
        if name.startswith('k_cv_adapted<') or name.startswith('k_cv_uniform<'):
            assert kernel_notes.waves_per_simd(k) >= (4 if 'uniform' in name else 3), name


def test_fixed_increment_adapted_kernels_hold_no_event_state():
    # the drawn path's event test in this kernel took 38 registers and 14% more time
    assert KERNELS['k_fixed<1, 0, 1, false>']['.vgpr_count'] <= 34
    assert KERNELS['k_fixed<1, 1, 1, false>']['.vgpr_count'] <= 40


@pytest.mark.parametrize('family', ['0', '1'])
@pytest.mark.parametrize('pois', ['false', 'true'])
def test_storing_uniform_kernels_keep_their_wavefronts(family, pois):
    # two to four components, beside the addresses of three stored arrays (a sixth
    # wavefront in four was no faster and its extra generator products 3% slower)
    for dim, waves in ((2, 8), (3, 6), (4, 5)):
        k = KERNELS['k_rng<%d, %s, 0, false, true, %s, -1>' % (dim, family, pois)]
        assert k['.private_segment_fixed_size'] == 0
        assert kernel_notes.waves_per_simd(k) >= waves
