"""What the module gk_torch is built for.  (A file of its own: the build runs it without the package, whose library is not there yet.)"""
import sysconfig


def built_for() -> str:
    """The ABI of this interpreter and its torch, as one line."""
    import torch
    return f"{sysconfig.get_config_var('SOABI')}, torch {torch.__version__} {torch.version.git_version}"
