"""Which loads of a kernel the device's range check covers: the vector offset is compared with the buffer's size, a scalar offset is not part of it."""
import os

ASM = """
_Z4probe_step_kernelv:
	buffer_load_dwordx4 v[2:5], v1, s[0:3], 0 offen offset:64
	buffer_load_ushort v6, off, s[4:7], 0
	buffer_load_dwordx4 v[8:11], v1, s[0:3], s9 offen
	buffer_store_dword v6, v7, s[0:3], 0 offen
	buffer_store_dword v6, v7, s[0:3], s10 offen offset:8
	s_endpgm
"""


def test_scalar_offsets_are_found():
    from msa_amd import build as B
    assert len(B.check_kernel_contracts(ASM, "probe_step_kernel", no_scalar_offset=True)) == 2
    assert B.check_kernel_contracts(ASM, "probe_step_kernel") == []


def test_one_token_of_the_delta_rule_has_none():
    """Its last turn of weight rows is partly behind the head's own, and for the last head behind the matrix."""
    from msa_amd import build as B
    assert B.CONTRACTS["seq_delta.hip"] == [("delta_step_kernel", {"no_scalar_offset": True})]
    asm = B._device_asm(os.path.join(B.CSRC, "seq_delta.hip"))
    assert B.check_kernel_contracts(asm, "delta_step_kernel", no_scalar_offset=True) == []
