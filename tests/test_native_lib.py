"""The C-ABI library loads and exports every symbol the header declares (CPU)."""
import ctypes
import os
import re
import subprocess

import pytest

from auto_infer_amd import _native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    names = set()
    for fn in os.listdir(os.path.join(ROOT, "include")):
        if fn.endswith(".h"):
            text = open(os.path.join(ROOT, "include", fn)).read()
            names |= set(re.findall(r"^\s*(?:const\s+)?\w+\*?\s+\*?(aia_\w+)\s*\(", text, re.M))
    return names


def test_header_declares_the_binding_table():
    assert declared_symbols() == set(_native.SIGNATURES)


def test_library_exports_all_declared_symbols():
    if not os.path.exists(_native.LIB_PATH):
        pytest.fail(f"library not built: {_native.LIB_PATH}")
    lib = ctypes.CDLL(_native.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(lib, name), name


def test_version_and_error_reporting_without_gpu():
    lib = _native.load()
    assert lib.aia_version() >= 100
    # argument validation happens before any device call
    rc = lib.aia_attn_workspace_bytes(4, 4, 3, 2, 128, 0, ctypes.byref(ctypes.c_int64()))
    assert rc == _native.AIA_ERR_INVALID
    assert "multiple" in _native.last_error()
    with pytest.raises(ValueError, match="multiple"):
        _native.check(rc, "aia_attn_workspace_bytes")


def test_workspace_query():
    out = ctypes.c_int64(0)
    _native.call("aia_attn_workspace_bytes", 16, 16, 16, 8, 128, 0, ctypes.byref(out))
    assert out.value > 0
    # sized for the range count asked for: the default 256 ranges of a
    # config-1 step need tens of MB, the maximum range count far more
    big = ctypes.c_int64(0)
    _native.call("aia_attn_workspace_bytes", 16, 16, 16, 8, 128, 16384, ctypes.byref(big))
    assert out.value < 64 << 20 < big.value


@pytest.mark.parametrize("hkv,group,d", [(1, 16, 512), (1, 7, 64), (2, 7, 64), (3, 8, 128),
                                         (4, 7, 128), (8, 8, 128), (300, 1, 128)])
@pytest.mark.parametrize("tokens", [256, 2048, 16384, 1 << 21])
def test_every_prefill_work_group_has_a_record_in_the_layout(hkv, group, d, tokens):
    """aia_attn_workspace_layout's one offset of the dealt work-groups holds
    a record (48 bytes) for every one a step can have: behind the (max, sum)
    pairs of the 512 row blocks that cut items may fill, those of a step with
    cut items (at most 512) in front of the partial values, all inside the
    workspace."""
    from auto_infer_amd import ops
    L = ops.workspace_layout(1, tokens, hkv * group, hkv, d)
    assert L["pf_unit_cap"] * hkv >= -(-tokens * group // 128) * hkv
    assert L["pfw"] >= L["pf_ml"] + 512 * 128 * 8
    assert L["pfw"] + 48 * 512 <= L["pf_o"]
    assert L["pfw"] + 48 * L["pf_unit_cap"] * hkv <= L["total"]
    assert L["pf_o"] + 512 * 128 * d * 2 <= L["total"]


def test_argument_validation_of_the_fused_kernels_without_gpu():
    """Bad arguments are rejected before any device call, with the mapped
    exception types."""
    lib = _native.load()
    vp = ctypes.c_void_p
    # qk norm + rope: head_dim other than 128 and 64 is unsupported
    rc = lib.aia_qk_norm_rope(vp(16), 1024, 4, 4, 2, 96, vp(16), 96, vp(16), 96, None, None,
                              ctypes.c_float(1e-6), None)
    assert rc == _native.AIA_ERR_UNSUPPORTED
    with pytest.raises(NotImplementedError, match="head_dim"):
        _native.check(rc, "aia_qk_norm_rope")
    # norm weights go together
    rc = lib.aia_qk_norm_rope(vp(16), 1024, 4, 4, 2, 128, vp(16), 128, vp(16), 128, vp(16), None,
                              ctypes.c_float(1e-6), None)
    assert rc == _native.AIA_ERR_INVALID and "together" in _native.last_error()
    # MTP compaction: gear limits
    for gear in (0, 65):
        rc = lib.aia_mtp_compact(*([vp(16)] * 4), 8, vp(16), vp(16), vp(16), vp(16), gear, 2, 8,
                                 vp(16), vp(16), 8, vp(16), vp(16), vp(16), None)
        assert rc == _native.AIA_ERR_INVALID and "gear" in _native.last_error()
    # paged GQA: the scale must be positive
    rc = lib.aia_paged_attention_gqa(vp(16), 2048, 128, vp(16), vp(16), vp(16), 16, vp(16),
                                     vp(16), 1, 1, 16, 8, 128, 16, 4, ctypes.c_float(0.0),
                                     vp(16), 2048, 128, None, None, 0, 0, 0, 0, vp(16), 1 << 20,
                                     None)
    assert rc == _native.AIA_ERR_INVALID and "scale" in _native.last_error()
    # the pool's slots must be addressable by the int32 slot_mapping
    rc = lib.aia_paged_attention_gqa(vp(16), 2048, 128, vp(16), vp(16), vp(16), 16, vp(16),
                                     vp(16), 1, 1, 16, 8, 128, 256, 1 << 23, ctypes.c_float(0.1),
                                     vp(16), 2048, 128, None, None, 0, 0, 0, 0, vp(16), 1 << 20,
                                     None)
    assert rc == _native.AIA_ERR_INVALID and "int32 slot range" in _native.last_error()
    rc = lib.aia_paged_attention_mla(vp(16), 16 * 576, 576, vp(16), vp(16), 16, vp(16), vp(16),
                                     1, 1, 16, 512, 64, 256, 1 << 23, ctypes.c_float(0.1),
                                     vp(16), 16 * 512, 512, 0, 0, vp(256), 1 << 20, None)
    assert rc == _native.AIA_ERR_INVALID and "int32 slot range" in _native.last_error()
    # the workspace must be 256-byte aligned
    rc = lib.aia_attn_plan(vp(256), vp(256), vp(256), 16, 16, 1, 1, 16, 8, 128, 0, vp(256 + 16),
                           1 << 30, None)
    assert rc == _native.AIA_ERR_INVALID and "256-byte" in _native.last_error()
    # absorbed-MLA latents: rows of 576 with 16-byte alignment
    rc = lib.aia_mla_kv_latent(vp(16), 500, 4, vp(16), ctypes.c_float(1e-6), vp(16), 64, vp(16),
                               64, vp(16), 576, None)
    assert rc == _native.AIA_ERR_INVALID and "576" in _native.last_error()
    rc = lib.aia_mla_kv_latent(vp(8), 576, 4, vp(16), ctypes.c_float(1e-6), vp(16), 64, vp(16),
                               64, vp(16), 576, None)
    assert rc == _native.AIA_ERR_INVALID
    rc = lib.aia_mla_q_latent(vp(16), 16 * 192, 192, 4, 0, vp(16), vp(16), 64, vp(16), 64,
                              vp(16), 16 * 576, 576, None)
    assert rc == _native.AIA_ERR_INVALID and "sizes" in _native.last_error()
    rc = lib.aia_mla_q_latent(vp(16), 16 * 192, 100, 4, 16, vp(16), vp(16), 64, vp(16), 64,
                              vp(16), 16 * 576, 576, None)
    assert rc == _native.AIA_ERR_INVALID and "alignment" in _native.last_error()
    # no tokens: nothing to do, whatever the pointers
    assert lib.aia_mla_q_latent(None, 0, 0, 0, 16, None, None, 0, None, 0, None, 0, 0, None) == 0


def test_public_limits_of_the_ops():
    """Names that programs route by stay: up to this many rows mla_v_up is the
    faster way."""
    from auto_infer_amd import ops
    assert ops.MLA_V_UP_MAX_ROWS >= 4096


def test_error_messages_are_per_thread():
    """aia_last_error() is thread local: two host threads failing with
    different arguments at the same time each read their own message."""
    import threading
    lib = _native.load()
    errs = []

    def worker(hq):
        out = ctypes.c_int64()
        for _ in range(2000):
            rc = lib.aia_attn_workspace_bytes(4, 4, hq, 2, 128, 0, ctypes.byref(out))
            msg = _native.last_error()
            if rc != _native.AIA_ERR_INVALID or f"num_q_heads {hq} " not in msg:
                errs.append((hq, rc, msg))
                return

    ts = [threading.Thread(target=worker, args=(hq,)) for hq in (3, 5, 7)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errs, errs[:3]


def _kernel_assembly(tmp_path, name):
    """Instructions (mnemonic, operands) of one kernel of the built library."""
    bins = "/opt/rocm/llvm/bin/"
    for tool in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump"):
        if not os.path.exists(bins + tool):
            pytest.skip(f"no {tool}")
    fat, out = str(tmp_path / "fat"), []
    subprocess.run([bins + "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", _native.LIB_PATH,
                    str(tmp_path / "copy")], check=True)
    # one bundle per source file, each aligned to a page behind its magic
    data = open(fat, "rb").read()
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)]
    for i, a in enumerate(starts):
        part, obj = str(tmp_path / f"part{i}"), str(tmp_path / f"obj{i}")
        open(part, "wb").write(data[a:(starts + [len(data)])[i + 1]])
        subprocess.run([bins + "clang-offload-bundler", "--type=o", "--unbundle", f"--input={part}",
                        f"--output={obj}", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        text = subprocess.run([bins + "llvm-objdump", "-d", "--mcpu=gfx950", obj], check=True,
                              capture_output=True, text=True).stdout
        inside = False
        for line in text.splitlines():
            if re.match(r"[0-9a-f]+ <", line):
                inside = name in line
            elif inside and line.strip():
                op, _, rest = line.split("//")[0].strip().partition(" ")
                out.append((op, [x.strip() for x in rest.split(",")]))
    return out


def _vgprs(operand):
    m = re.fullmatch(r"[-|]*v(\d+)\|?", operand) or re.fullmatch(r"v\[(\d+):(\d+)\]", operand)
    if not m:
        return set()
    return set(range(int(m[1]), int(m[m.lastindex]) + 1))


def test_mla_score_mfmas_have_their_wait_states(tmp_path):
    """The MLA prefill kernel issues QK^T as inline assembly, which the
    compiler's hazard recogniser does not see as MFMAs.  In the built kernel:
    no VALU instruction writes an operand of one within two wait states in
    front of it; between the links of a chain nothing else reads or writes
    the accumulator; and behind the last link its first other use is 11 wait
    states away (an 8-pass MFMA's), an MFMA in between counting as its 8."""
    code = _kernel_assembly(tmp_path, "mla_prefill_kernel")
    assert code
    states = [int(a[0], 0) + 1 if op == "s_nop" else 8 if op.startswith("v_mfma") else 1 for op, a in code]
    links = [i for i, (op, a) in enumerate(code) if op.startswith("v_mfma") and _vgprs(a[0])]
    chains = sum(code[i][1][3] == "0" for i in links)
    assert chains >= 3 and len(links) == 36 * chains       # a first, a plain and a masked step
    for n, i in enumerate(links):
        acc, operands = _vgprs(code[i][1][0]), set().union(*map(_vgprs, code[i][1]))
        waited, j = 0, i - 1
        while waited < 2:
            op, a = code[j]
            if op.startswith("v_") and not op.startswith("v_mfma"):
                written = _vgprs(a[0]) | (_vgprs(a[1]) if "swap" in op else set())
                assert not written & operands, (code[j], code[i])
            waited, j = waited + states[j], j - 1
        last = n + 1 == len(links) or code[links[n + 1]][1][3] == "0"
        stop = len(code) if last else links[n + 1]
        waited, j = 0, i + 1
        while j < stop and (not last or waited < 11):
            op, a = code[j]
            assert not set().union(*map(_vgprs, a)) & acc, (code[i], code[j], waited)
            waited, j = waited + states[j], j + 1
