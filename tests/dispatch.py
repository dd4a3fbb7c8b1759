"""The kernels that an entry point launches for a call, without a GPU: the entry point itself runs on a recording
context (nh_runtime.h), which notes its launches in place of making them.  Pointers are made-up device addresses."""
import ctypes as C

import nemotron_hip as NH

CUS, LDS = 256, 163840  # an MI355X
X, W, S, OUT, WS, BIAS, W2, S2 = (i << 40 for i in range(1, 9))  # apart and aligned


class Recorder:
    def __init__(self, cus=CUS, lds=LDS):
        self.lib = NH.lib()
        self.lib.nh_record_context.restype = C.c_void_p
        self.lib.nh_record_context.argtypes = [C.c_int, C.c_size_t]
        self.lib.nh_record_take.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int]
        self.lib.nh_record_free.argtypes = [C.c_void_p]
        self.ctx = self.lib.nh_record_context(cus, lds)
        assert self.ctx

    def close(self):
        self.lib.nh_record_free(self.ctx)

    def launches(self, name, *args):
        """[(kernel name without nh_ and _kernel, grid width, grid height)] of one call."""
        NH.call(name, self.ctx, *args)
        names, gx, gy = (C.c_char_p * 64)(), (C.c_uint32 * 64)(), (C.c_uint32 * 64)()
        n = self.lib.nh_record_take(self.ctx, names, gx, gy, 64)
        assert n <= 64
        return [(names[i].decode()[3:-7], gx[i], gy[i]) for i in range(n)]

    def kernels(self, name, *args):
        return [k for k, _, _ in self.launches(name, *args)]

    def linear(self, m, n, k, x_dtype=NH.BF16, out_dtype=NH.BF16, x=X, out=OUT, xq_out=None, sx_out=None):
        ws = NH.lib().nh_linear_w8a8_workspace_size(m, k)
        return self.kernels("nh_linear_w8a8", x, x_dtype, W, S, None, m, n, k, out, out_dtype, WS, ws, xq_out, sx_out,
                            None, None)

    def gemm_ta(self, m, n, k, out_dtype=NH.BF16, out=OUT):
        return self.kernels("nh_gemm_w8a8_ta", X, S, W, S, None, m, n, k, out, out_dtype, None)

    def w4a8(self, m, n, k, x_dtype=NH.BF16, workspace=True, x=X, out=OUT):
        ws = NH.lib().nh_linear_w4a8_workspace_size(m, n, k)
        return self.kernels("nh_linear_w4a8", x, x_dtype, W, 0.01, 8, None, m, n, k, out, NH.BF16, WS if workspace else None,
                            ws if workspace else 0, None, None)

    def mlp(self, m, hidden, inter, x_dtype=NH.BF16, out_dtype=NH.BF16):
        ws = NH.lib().nh_mlp_w8a8_workspace_size(m, hidden, inter)
        return self.kernels("nh_mlp_w8a8", X, x_dtype, W, S, BIAS, W2, S2, BIAS, m, hidden, inter, OUT, out_dtype, WS, ws, None,
                            None)
