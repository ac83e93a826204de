"""build_lib.py on the CPU: what the C-ABI library's link depends on (the
compilers are replaced; nothing is built)."""
import importlib.util

import pytest

import build_lib


@pytest.fixture
def recorded(monkeypatch, tmp_path):
    """build() with its compile and link steps recorded instead of run."""
    steps = []
    monkeypatch.setattr(build_lib, 'BUILD', tmp_path / 'obj')
    monkeypatch.setattr(build_lib, '_compile', lambda unit, verbose: steps.append('unit') or unit[1])
    monkeypatch.setattr(build_lib, '_link', lambda objs, verbose: steps.append('library'))
    monkeypatch.setattr(build_lib, '_link_native', lambda obj, verbose: steps.append('native'))
    return steps


def test_library_is_linked_when_the_native_module_cannot_be_compiled(recorded, monkeypatch):
    def fail(verbose):
        raise RuntimeError('no Python.h')
    monkeypatch.setattr(build_lib, '_compile_native', fail)
    with pytest.raises(RuntimeError, match='no Python.h'):
        build_lib.build(jobs=2)
    assert recorded[-1] == 'library' and recorded.count('unit') == len(build_lib._units())


def test_library_without_torch(recorded, monkeypatch):
    real = importlib.util.find_spec
    monkeypatch.setattr(importlib.util, 'find_spec', lambda name, *a: None if name == 'torch' else real(name, *a))
    monkeypatch.setattr(build_lib, '_compile_native', lambda verbose: pytest.fail('native.cpp compiled without torch'))
    assert build_lib.build(jobs=2) == build_lib.OUT
    assert recorded[-1] == 'library'


def test_native_module_follows_the_library(recorded, monkeypatch):
    monkeypatch.setattr(build_lib, '_compile_native', lambda verbose: 'native.o')
    build_lib.build(jobs=2)
    assert recorded[-2:] == ['library', 'native']
