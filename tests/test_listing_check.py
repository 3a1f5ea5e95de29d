"""The check of hand-placed MFMAs finds a planted break of each of its rules, and nothing in clean code."""
import pytest

from simplical_attn_amd import listing_check

CLEAN = """k_kernel:
\tv_accvgpr_write_b32 a192, v9
\tds_read_b128 v[4:7], v9
\tv_mul_f32_e32 v1, v2, v3
\ts_waitcnt lgkmcnt(0)
\tv_mov_b32_e32 v8, 0
\t;;#ASMSTART
\tv_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], a[0x80:0x83], v[32:47]
\tv_mfma_f32_32x32x16_bf16 a[0:15], v[4:7], v[0:3], a[0:15]
\tv_mfma_f32_32x32x16_bf16 a[16:31], v[4:7], v[0:3], a[16:31]
\tv_accvgpr_read_b32 v9, a[40:40]
\t;;#ASMEND
\tv_exp_f32_e32 v16, v16
"""


@pytest.mark.parametrize("old,new,rule", [
    ("", "", None),
    ("ds_read_b128 v[4:7]", "ds_read_b128 a[4:7]", 1),
    ("v_accvgpr_write_b32 a192", "v_accvgpr_write_b32 a191", 1),
    ("v_mov_b32_e32 v8, 0", "v_mov_b32_e32 v4, 0", 2),
    ("\tv_mfma_f32_32x32x16_bf16 a[16:31], v[4:7], v[0:3], a[16:31]\n", "", 3),
    ("v_mov_b32_e32 v8, 0", "s_mov_b32 m0, s4", 4),
])
def test_planted_breaks(old, new, rule):
    bad, found = listing_check.violations(CLEAN.replace(old, new, 1).splitlines(), "k_kernel", 192)
    assert found == 1
    assert {b[0] for b in bad} == (set() if rule is None else {rule})


@pytest.mark.parametrize("name,register", [("_Z20mfma_fwd_lone_kernelI8ElemBF16Li128ELb0EEv", 150), ("_Z20mfma_fwd_lone_kernelI7ElemF16Li64ELb1EEv", 95),
                                           ("_Z18mfma_bwd_kv_kernelI7ElemF16Li64EEv", 191), ("_Z23mfma_bwd_kp_lone_kernelI7ElemF16Li64EEv", 255)])
def test_every_owned_register_is_watched(name, register):
    """The table that the build uses finds an instruction of the compiler's in any register that a kernel owns."""
    from simplical_attn_amd import build
    code = CLEAN.replace("k_kernel", name).replace("a192, v9", "a%d, v9" % register)
    found = {}
    for source, kernels in build.HAND_PLACED.items():
        for pattern, owned in kernels:
            found.setdefault(source, []).extend(r[0] for r in listing_check.violations(code.splitlines(), pattern, owned)[0])
    hits = [source for source, rules in found.items() if rules]
    assert len(hits) == 2 and all(found[s] == [1] for s in hits)       # the bf16 and the fp16 source of that kernel
