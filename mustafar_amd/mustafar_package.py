"""Drop-in for the reference's `mustafar_package` extension (kernel/kernel_wrapper/pybind.cpp:7-10,
mustafar_wrapper.cu:19-263): same positional arguments, same checks (RuntimeError), same output
shape [Batch_Size, 8, M_Global] fp16, launched on the current stream without synchronising."""
from . import ops
from ._lib import host


def mustafar_key_formulation(bmp, NZ, idx, NZ_Offset, B, M_Global, K_Global, Batch_Size, num_key_value_groups):
    """C[bq, n, m] = sum_k Ktilde[bq // groups][m, k] * B[bq, n, k];  B: [Batch_Size, 8, K_Global]."""
    return host().key_formulation(bmp, NZ, idx, NZ_Offset, B, int(M_Global), int(K_Global), int(Batch_Size),
                                  int(num_key_value_groups))


def mustafar_value_formulation(bmp, NZ, idx, NZ_Offset, B, Reduction_Workspace, M_Global, K_Global, Batch_Size,
                               num_key_value_groups):
    """C[bq, n, m] = sum_k Vtilde[bq // groups][k, m] * B[bq, n, k];  B: [Batch_Size, 8, K_Global].

    Reduction_Workspace is accepted for signature compatibility (the reference passes a one-element
    dummy); the fp32 split partials live in the package's own scratch tensor."""
    return ops._call(host().value_formulation, None, B.device, None, bmp, NZ, idx, NZ_Offset, B, int(M_Global), int(K_Global),
                     int(Batch_Size), int(num_key_value_groups))
