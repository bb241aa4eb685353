"""The argument structures filled in one call hold, field by field, what was packed."""

import ctypes

import pytest

from geometric_nn_ops_torch import _lib


@pytest.mark.parametrize(("cls", "pack"), [(_lib.TriAttnArgs, _lib.pack_triattn),
                                           (_lib.TriAttnBwdArgs, _lib.pack_triattn_bwd),
                                           (_lib.TrimulArgs, _lib.pack_trimul)])
def test_packed_fields(cls, pack):
    values, want = [], {}
    for name, typ in cls._fields_:
        n = getattr(typ, "_length_", 1)
        part = [len(values) + i + 1 for i in range(n)]
        want[name] = part
        values += part
    args = cls()
    pack(args, 0, *values)
    for name, typ in cls._fields_:
        got = getattr(args, name)
        assert (list(got) if hasattr(typ, "_length_") else [got]) == want[name], name
    pack(args, 0, *[0] * len(values))
    assert bytes(args) == bytes(ctypes.sizeof(cls))


def test_weight_pointers_follow_the_structure():
    """The trimul call packs its weights in _WEIGHT_KEYS order."""
    from geometric_nn_ops_torch.triangle._kernels.trimul import _WEIGHT_KEYS

    names = [n for n, _ in _lib.TrimulArgs._fields_]
    first = names.index("ln_in_w")
    assert [n.replace("ln_", "norm_").replace("_b", "_bias").replace("_w", "_weight")
            for n in names[first:first + len(_WEIGHT_KEYS)]] == list(_WEIGHT_KEYS)
