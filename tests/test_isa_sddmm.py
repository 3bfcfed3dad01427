"""The DPP wait states of test_isa.py for the panel form of the sampled product,
whose steps use the same inline assembly."""
from test_isa import HIPCC, device_asm, dpp_hazards, functions, pytestmark  # noqa: F401


def test_panel_sddmm_dpp_wait_states(device_asm):  # noqa: F811
    fns = functions(device_asm, "panel_sddmm_kernel")
    assert len(fns) >= 7, sorted(fns)
    for name, body in fns.items():
        assert sum("_dpp " in ln for ln in body) > 100
        bad = dpp_hazards(body)
        assert not bad, (name, bad[:5])
