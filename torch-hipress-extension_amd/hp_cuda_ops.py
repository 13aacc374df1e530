"""Host-side mirror of the reference's kernel-driver layer.

The nine functions below carry the names, argument order and argument meaning
of the `hp_cuda_*` free functions the reference declares in hp_cuda.cpp:18-102
and defines in hp_cuda_kernel.cu; each forwards to the C-ABI entry point of
libhpx.so that replaces it.  Where the reference takes std::vector<float*> a
list of CUDA-device torch tensors (or raw device addresses) is taken, and the
trailing `stream` is a torch.cuda.Stream, a raw hipStream_t address, or None
for the current stream.

Like the reference drivers they report a body failure by printing and carry on
(hp_cuda_kernel.cu:63, :90-92, :115-117, :153-155); unlike them they also
return the code.  `seeds` is an addition: the reference draws its RNG seed from
the wall clock inside the body and cannot be seeded from outside.
"""
import torch

from . import _capi


def _calls():
    """The native module that lays the argument lists out and makes the calls (csrc/hp_calls_module.cpp)."""
    global _native
    if _native is None:
        _capi.load()
        _native = _capi.load_extension("_hp_calls")
    return _native


_native = None


def _stream(stream):
    return stream.cuda_stream if isinstance(stream, torch.cuda.Stream) else stream


def _report(rc, what):
    if rc:
        print(f"Call {what} failed, ret = {rc}. {_capi.last_error()}", flush=True)
    return rc


def hp_cuda_tbq(to_compress_floats, to_compress_float_sizes, residual_floats, residual_float_sizes,
                out_uint8_ts, out_uint8_t_sizes, thresholds, stream=None):
    """hp_cuda_kernel.cu:120-158; waits for the stream like the reference (:157)."""
    return _report(_calls().tbq(to_compress_floats, to_compress_float_sizes, residual_floats, out_uint8_ts, thresholds,
                                _stream(stream)), "tbq_body")


def hp_cuda_tbqr(out_floats, out_float_sizes, in_uint8_ts, in_uint8_t_sizes, thresholds, is_add_tos, stream=None):
    """hp_cuda_kernel.cu:161-198; waits for the stream like the reference (:197)."""
    return _report(_calls().tbqr(out_floats, out_float_sizes, in_uint8_ts, thresholds, is_add_tos, _stream(stream)), "tbq_r_body")


def hp_cuda_terngrad(in_floats, in_float_sizes, out_uint8_ts, out_uint8_t_sizes, bitwidths, enable_randoms,
                     stream=None, seeds=None):
    """hp_cuda_kernel.cu:30-65."""
    return _report(_calls().terngrad(in_floats, in_float_sizes, out_uint8_ts, out_uint8_t_sizes, bitwidths, enable_randoms,
                                     _stream(stream), seeds), "terngrad_body")


def hp_cuda_terngradr(out_floats, out_float_sizes, in_uint8_ts, in_uint8_t_sizes, is_add_tos, stream=None):
    """hp_cuda_kernel.cu:200-230."""
    return _report(_calls().terngradr(out_floats, out_float_sizes, in_uint8_ts, in_uint8_t_sizes, is_add_tos, _stream(stream)),
                   "terngrad_r_body")


def hp_cuda_gd(in_floats, Ns, residuals, residual_sizes, out_uint8_ts, sample_rates, drop_ratios,
               stream=None, seeds=None):
    """hp_cuda_kernel.cu:67-94."""
    return _report(_calls().gd(in_floats, Ns, residuals, out_uint8_ts, sample_rates, drop_ratios, _stream(stream), seeds), "gd_body")


def hp_cuda_gdr(in_uint8_ts, in_uint8_t_sizes, out_floats, out_float_sizes, is_add_tos, stream=None):
    """hp_cuda_kernel.cu:96-118."""
    return _report(_calls().gdr(in_uint8_ts, in_uint8_t_sizes, out_floats, out_float_sizes, is_add_tos, _stream(stream)), "gdr_body")


def hp_cuda_powersgd_encode1(grads, residuals, Qs, Ms, Ps, stream=None):
    """hp_cuda_kernel.cu:232-255: M[:N] = grad + residual, P = M Q."""
    return _report(_calls().powersgd_encode1(grads, residuals, Qs, Ms, Ps, _stream(stream)), "powersgd encode1")


def hp_cuda_powersgd_encode2(Ps, Ms, Qs, stream=None):
    """hp_cuda_kernel.cu:257-276: P = orth(P), Q = M^T P."""
    return _report(_calls().powersgd_encode2(Ps, Ms, Qs, _stream(stream)), "powersgd encode2")


def hp_cuda_powersgd_decode(Ps, Qs, Ms, residuals, grads, stream=None):
    """hp_cuda_kernel.cu:278-301: M = P Q^T, residual = grad - M[:N], grad = M[:N]."""
    return _report(_calls().powersgd_decode(Ps, Qs, Ms, residuals, grads, _stream(stream)), "powersgd decode")
