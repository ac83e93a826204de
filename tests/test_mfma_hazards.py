"""The build's check of the wait states around inline-assembly MFMAs, on small
assembly texts (CPU only)."""
import pytest

from mfma_hazards import hazards

MFMA = 'v_mfma_i32_16x16x64_i8 a[0:3], v[4:7], v[8:11], a[0:3]'


def _text(body, scratch=0):
    lines = '\n'.join(line if line.endswith(':') else '\t' + line for line in body)
    return f'kernel_a:\n{lines}\n\ts_endpgm\n; ScratchSize: {scratch}\n'


@pytest.mark.parametrize('body', [
    ['ds_read_b128 v[4:7], v20', 's_waitcnt lgkmcnt(0)', MFMA],            # the compiler counts LDS reads itself
    ['v_mov_b32_e32 v4, v1', 's_nop 1', MFMA],                             # two wait states
    ['v_mov_b32_e32 v3, v4', MFMA],                                        # another register
    ['v_accvgpr_write_b32 a0, v1', 's_nop 7', MFMA],
    [MFMA, 's_nop 15', 's_nop 1', 'v_accvgpr_read_b32 v1, a3'],            # eighteen
    [MFMA, 'v_mfma_i32_16x16x64_i8 a[0:3], v[4:7], v[8:11], a[0:3]'],      # the pipeline orders MFMAs
    [MFMA, 'v_accvgpr_read_b32 v1, a4'],
    ['v_cmpx_lt_i32_e32 v1, v2', 's_nop 3', MFMA],
    ['v_readfirstlane_b32 s4, v4', MFMA],
])
def test_accepted(body):
    assert hazards(_text(body), 'kernel') == []


@pytest.mark.parametrize('body', [
    ['v_mov_b32_e32 v11, v1', MFMA],
    ['v_accvgpr_read_b32 v4, a9', 's_nop 0', MFMA],                        # an AGPR copied back just before
    ['v_add_u32_e32 v8, v1, v2 ; a comment', 's_add_i32 s0, s0, 1', MFMA],
    ['v_accvgpr_write_b32 a2, v1', MFMA],
    ['v_permlane32_swap_b32_e32 v1, v5', MFMA],                            # writes both operands
    ['v_cmpx_lt_i32_e32 v1, v2', 's_nop 2', MFMA],
    [MFMA, 's_nop 15', 'v_accvgpr_read_b32 v1, a3'],
    [MFMA, 's_nop 7', 'global_store_dwordx4 v20, a[0:3], s[2:3]'],
    # around a loop's end, and over a taken branch
    ['.LBB0_1:', MFMA, 's_nop 15', 's_nop 7', 'v_mov_b32_e32 v7, v1', 's_cbranch_scc1 .LBB0_1'],
    ['v_mov_b32_e32 v5, v1', 's_cbranch_vccz .LBB0_2', 's_nop 7', '.LBB0_2:', MFMA],
    [MFMA, 's_cbranch_scc1 .LBB0_3', 's_nop 15', 's_nop 15', '.LBB0_3:', 'v_accvgpr_read_b32 v1, a0'],
])
def test_hazards_are_found(body):
    assert hazards(_text(body), 'kernel')


def test_scratch_and_missing_kernels_are_found():
    assert 'scratch' in hazards(_text([MFMA], scratch=8), 'kernel')[0]
    assert 'no function' in hazards(_text([MFMA]), 'other')[0]
