"""Whether a submodule's work may be done apart from its call."""

from torch.nn.modules import module as _nn


def unhooked(module, cls) -> bool:
    """Whether calling ``module`` is ``cls.forward`` and nothing else: no hook of its
    own or of all modules, no other class or function in its place."""
    return (
        type(module) is cls
        and "forward" not in vars(module)
        and not (
            module._forward_pre_hooks
            or module._forward_hooks
            or module._backward_pre_hooks
            or module._backward_hooks
            or _nn._has_any_global_hook()
        )
    )
