"""The C headers against the version numbers that bindings compare at load time, and against the argument lists of the bindings."""
import hashlib
import os
import re
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# version of the mixer library's interface -> digest of its prototypes.  A prototype that is added, removed or changed needs the next number and its digest here.
MIX_PROTOTYPES = {6: "87c980474bb9d971", 7: "fa10166b1c0ce953"}


def _prototypes(name):
    with open(os.path.join(ROOT, "include", name)) as f:
        text = re.sub(r"/\*.*?\*/", " ", f.read(), flags=re.S)
    text = "\n".join(l for l in text.splitlines() if not l.lstrip().startswith("#"))
    return {m.group(2): (m.group(1), [" ".join(a.split()) for a in m.group(3).split(",")] if m.group(3).strip() != "void" else [])
            for m in re.finditer(r"([\w ]+?\*?)\s*\b(exl3_\w+)\s*\(([^()]*)\)\s*;", text)}


def test_mixer_version_number_follows_its_prototypes():
    with open(os.path.join(ROOT, "include", "exl3_mix.h")) as f:
        version = int(re.search(r"#define EXL3_MIX_ABI_VERSION (\d+)", f.read()).group(1))
    from exllamav3_amd import _lib
    text = "\n".join(f"{ret.strip()} {name}({','.join(args)})" for name, (ret, args) in sorted(_prototypes("exl3_mix.h").items()))
    digest = hashlib.sha256(text.encode()).hexdigest()[:16]
    assert version == _lib.MIX_ABI_VERSION
    assert MIX_PROTOTYPES.get(version) == digest, f"prototypes of exl3_mix.h changed (digest {digest}): raise EXL3_MIX_ABI_VERSION"


def test_segmented_recurrence_keeps_its_argument_list():
    args = _prototypes("exl3_mix.h")["exl3_mix_gla_segmented"][1]
    assert len(args) == 28 and args[-4:] == ["float* seg_state", "float* seg_decay", "int dtype", "void* stream"]


@pytest.mark.parametrize("header,declare", [("exl3_mix.h", "_declare_mix"), ("exl3_hip.h", "_declare")])
def test_bindings_pass_as_many_arguments_as_the_header_names(header, declare):
    from exllamav3_amd import _lib

    class Recorder:
        def __getattr__(self, name):
            fn = type("Fn", (), {"argtypes": None, "restype": None})()
            setattr(self, name, fn)
            return fn
    lib, protos = Recorder(), _prototypes(header)
    getattr(_lib, declare)(lib)
    declared = {n: f.argtypes for n, f in vars(lib).items() if f.argtypes is not None}
    assert len(declared) > 40
    wrong = {n: (len(a), len(protos[n][1])) for n, a in declared.items() if n in protos and len(a) != len(protos[n][1])}
    assert not wrong
