"""What stands between a module's call and its forward()."""
from __future__ import annotations

from torch.nn.modules import module as _nn


def plain(cls: type, *modules) -> bool:
    """True where calling any of `modules` is cls.forward and nothing else: no
    subclass or other module in its place, no forward of the object's own, no
    hook. Kernels that do the work of several modules ask before they pass
    them by."""
    if (_nn._global_forward_hooks or _nn._global_forward_pre_hooks or
            _nn._global_backward_hooks or _nn._global_backward_pre_hooks):
        return False
    for m in modules:
        if type(m) is not cls:
            return False
        d = m.__dict__
        if ("forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"] or
                d["_backward_hooks"] or d["_backward_pre_hooks"]):
            return False
    return True


def untouched(names, *modules) -> bool:
    """True where no object of `modules` has methods of its own of these
    names: those that are called in place of forward()."""
    return not any(name in m.__dict__ for m in modules for name in names)
