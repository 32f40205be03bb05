"""Parts name the kernel libraries that they launch, so that a model's are built before its first step."""
import importlib
import inspect
import pkgutil

import ginfer_amd.parts
from ginfer_amd.parts.base import Part


def _parts():
    for m in pkgutil.iter_modules(ginfer_amd.parts.__path__):
        importlib.import_module("ginfer_amd.parts." + m.name)
    todo, seen = [Part], []
    while todo:
        for cls in todo.pop().__subclasses__():
            if cls not in seen:
                seen.append(cls)
                todo.append(cls)
    return [c for c in seen if c.__module__.startswith("ginfer_amd.parts.")]


def test_parts_whose_products_may_run_over_tiles_name_that_library():
    users = [c for c in _parts() if "parts_ok=" in inspect.getsource(c) or "gated_linear(" in inspect.getsource(c)]
    assert len(users) >= 8
    for cls in users:
        assert '"gemm_tiles"' in inspect.getsource(cls.kernel_modules), cls.__name__
