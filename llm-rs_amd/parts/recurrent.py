"""Recurrent mixers: each keeps a state of fixed size per request (in the request's slot, 32-bit), reads it at the
start of a step's portion and leaves it for the next; nothing is paged.

"mingru"(hidden_size, width): gate z = sigmoid(Wz x + bz), candidate c = g(Wc x + bc) with g(u) = u + 1/2 for u >= 0
and sigmoid(u) below; s_t = (1 - z) s_{t-1} + z c; h += Wo (s_t * silu(Wg x)).  One product gives the three
projections' 32-bit sums; the scan kernel does the rest in 32-bit and writes the gated state in the activation type.

"mamba1"(hidden_size, inner, state, conv, dt_rank): the selective scan.  [x | g] = Win h (32-bit sums); x <-
silu(causal conv over `conv` taps, last tap the current token); [d | B | C] = Wx x; step = softplus(Wdt d + bdt);
S[c, n] <- exp(step_c A[c, n]) S[c, n] + step_c x_c B_n with A = -exp(A_log); y_c = sum_n S[c, n] C_n + D_c x_c;
h += Wo (y * silu(g)).  The request's state is S and the convolution's last conv - 1 inputs.

"gated_unit"(hidden_size, width, blocks, conv): a gated linear recurrent unit behind a convolution.  y = gelu(Wy h + by)
in gelu's tanh form; u = causal conv over `conv` taps of Wx h + bx, with a bias and no activation; u falls into `blocks` equal
parts, each with square matrices of its own for r = sigmoid(Wr_b u_b + br_b) and i = sigmoid(Wi_b u_b + bi_b);
log a = -8 r softplus(lambda), S_t = a S_(t-1) + sqrt(1 - a^2) i u, also for the first token (from S = 0); h += Wo (S * y).  The
request's state is S and the convolution's last conv - 1 inputs.
"""
from __future__ import annotations

import torch

from ..cache.spec import FixedState
from ..kernels import EPI_ACCUM_F32, EPI_STORE, EPI_STORE_F32, kernels
from .base import Mixer, TensorSpec, place, register_mixer


def _leaves(defaults: dict, given) -> dict:
    return {**defaults, **(given or {})}


class MinGRU(Mixer):
    graph_safe = True

    def __init__(self, spec, dtype):
        super().__init__(spec, dtype)
        p = spec.params
        self.hidden, self.width = int(p["hidden_size"]), int(p["width"])
        leaves = _leaves({"gate": "z", "gate_bias": "z.b", "candidate": "x", "candidate_bias": "x.b", "out_gate": "g", "out": "o"}, p.get("names"))
        self.names = {k: self.name(v) for k, v in leaves.items()}
        self.w_in = self.w_o = self.bias_z = self.bias_c = None
        self.step_in_products = self.hidden % 8 == 0 and self.width % 8 == 0          # (rows of whole 16-byte pieces, eights of channels)

    def tensors(self):
        n, W, H = self.names, self.width, self.hidden
        return {n["gate"]: TensorSpec((W, H)), n["gate_bias"]: TensorSpec((W,)), n["candidate"]: TensorSpec((W, H)),
                n["candidate_bias"]: TensorSpec((W,)), n["out_gate"]: TensorSpec((W, H)), n["out"]: TensorSpec((H, W))}

    def load(self, tensors, device):
        n = self.names
        get = lambda key: place(tensors[n[key]], device, self.dtype)
        self.w_in = torch.cat([get("gate"), get("candidate"), get("out_gate")], dim=0).contiguous()
        self.w_o = get("out")
        self.bias_z = place(tensors[n["gate_bias"]], device, torch.float32)
        self.bias_c = place(tensors[n["candidate_bias"]], device, torch.float32)

    def export(self):
        n, W = self.names, self.width
        w = self.w_in.cpu()
        return {n["gate"]: w[:W].contiguous(), n["candidate"]: w[W:2 * W].contiguous(), n["out_gate"]: w[2 * W:].contiguous(),
                n["out"]: self.w_o.cpu(), n["gate_bias"]: self.bias_z.cpu(), n["candidate_bias"]: self.bias_c.cpu()}

    def cache_need(self):
        return FixedState((self.width,), torch.float32)

    def forward(self, ctx, x, h, cache):
        k = kernels()
        T = x.shape[0]
        # (up to 16 requests of one token: the product advances the state itself)
        if self.step_in_products and k.products_step_mixers(T, ctx.n_entries, ctx.longest, self.dtype,
                                                                  (x, self.w_in, self.bias_z, self.bias_c, cache.state)):
            gated = ctx.workspace("mingru.gated", (T, self.width), self.dtype)
            k.mingru_product_step(x, self.w_in, self.bias_z, self.bias_c, cache.state, ctx.slots, self.width, gated)
            k.gemm(gated, self.w_o, h, EPI_ACCUM_F32, ctx.gemm_workspace(gated, self.w_o))
            ctx.note_left(h, None)
            return
        sums = ctx.workspace("mingru.sums", (T, 3 * self.width), torch.float32)
        k.gemm(x, self.w_in, sums, EPI_STORE_F32, ctx.gemm_workspace(x, self.w_in))
        gated = ctx.workspace("mingru.gated", (T, self.width), self.dtype)
        need = k.scan_carry_floats(T, ctx.n_entries, ctx.longest, 2 * self.width)
        carry = ctx.workspace("scan.carry", (need,), torch.float32) if need else None
        k.mingru_scan(sums, self.bias_z, self.bias_c, cache.state, ctx.q_starts, ctx.slots, self.width, gated, ctx.longest, carry)
        k.gemm(gated, self.w_o, h, EPI_ACCUM_F32, ctx.gemm_workspace(gated, self.w_o))
        ctx.note_left(h, None)


class Mamba1(Mixer):
    graph_safe = True

    def __init__(self, spec, dtype):
        super().__init__(spec, dtype)
        p = spec.params
        self.hidden, self.inner, self.n_state = int(p["hidden_size"]), int(p["inner"]), int(p["state"])
        self.taps, self.dt_rank = int(p["conv"]), int(p["dt_rank"])
        if self.taps < 1:
            raise ValueError("the convolution has at least one tap")
        leaves = _leaves({"in": "in", "conv": "conv", "conv_bias": "conv.b", "x": "x", "dt": "dt", "dt_bias": "dt.b",
                          "A_log": "A_log", "D": "D", "out": "o"}, p.get("names"))
        self.names = {k: self.name(v) for k, v in leaves.items()}
        self.w_in = self.w_x = self.w_dt = self.w_o = None
        self.conv = self.conv_bias = self.dt_bias = self.A = self.A_log = self.D = None
        # (four taps and 16 states, as most have; rows of whole 16-byte pieces, sixteens of channels)
        self.step_in_products = (self.taps == 4 and self.n_state == 16 and self.hidden % 8 == 0 and self.dt_rank % 8 == 0 and self.inner % 16 == 0)

    def tensors(self):
        n, C, H, N, R = self.names, self.inner, self.hidden, self.n_state, self.dt_rank
        return {n["in"]: TensorSpec((2 * C, H)), n["conv"]: TensorSpec((C, self.taps), "normal:0.0:0.3"), n["conv_bias"]: TensorSpec((C,)),
                n["x"]: TensorSpec((R + 2 * N, C)), n["dt"]: TensorSpec((C, R), "normal:0.0:0.1"), n["dt_bias"]: TensorSpec((C,), "normal:-2.0:0.5"),
                n["A_log"]: TensorSpec((C, N), "normal:0.0:0.5"), n["D"]: TensorSpec((C,), "norm"), n["out"]: TensorSpec((H, C))}

    def load(self, tensors, device):
        n = self.names
        get = lambda key: place(tensors[n[key]], device, self.dtype)
        get32 = lambda key: place(tensors[n[key]], device, torch.float32)
        self.w_in, self.w_x, self.w_dt, self.w_o = get("in"), get("x"), get("dt"), get("out")
        self.conv, self.conv_bias, self.dt_bias, self.D = get32("conv"), get32("conv_bias"), get32("dt_bias"), get32("D")
        self.A_log = get32("A_log")
        self.A = (-torch.exp(self.A_log)).t().contiguous()      # 32-bit, once; [state, inner] as the scan reads it

    def export(self):
        n = self.names
        return {n["in"]: self.w_in.cpu(), n["x"]: self.w_x.cpu(), n["dt"]: self.w_dt.cpu(), n["out"]: self.w_o.cpu(),
                n["conv"]: self.conv.cpu(), n["conv_bias"]: self.conv_bias.cpu(), n["dt_bias"]: self.dt_bias.cpu(),
                n["D"]: self.D.cpu(), n["A_log"]: self.A_log.cpu()}

    def step_weight_bytes(self, seen):
        seen.add(self.A_log.data_ptr())      # a step reads A, not its logarithm
        return super().step_weight_bytes(seen)

    def cache_need(self):
        # one row per request: the scan's state [state, inner], then the convolution's last inputs [conv - 1, inner]
        return FixedState((self.inner * self.n_state + (self.taps - 1) * self.inner,), torch.float32)

    def forward(self, ctx, x, h, cache):
        k = kernels()
        T, C, N, R = x.shape[0], self.inner, self.n_state, self.dt_rank
        sums = ctx.workspace("mamba.sums", (T, 2 * C), torch.float32)
        scan_state, conv_state = cache.state[:, :C * N], cache.state[:, C * N:]
        xc = ctx.workspace("mamba.x", (T, C), self.dtype)
        dbc = ctx.workspace("mamba.dbc", (T, R + 2 * N), self.dtype)
        y = ctx.workspace("mamba.y", (T, C), self.dtype)
        # (up to 16 requests of one token: the products convolve and, of few states, advance the state themselves)
        in_products = self.step_in_products and k.products_step_mixers(T, ctx.n_entries, ctx.longest, self.dtype,
                                                                        (x, self.w_in, self.conv, self.conv_bias, cache.state, self.w_dt))
        if in_products:
            k.conv_product_step(x, self.w_in, sums, self.conv, self.conv_bias, conv_state, ctx.slots, C, xc)
        else:
            k.gemm(x, self.w_in, sums, EPI_STORE_F32, ctx.gemm_workspace(x, self.w_in))
            k.causal_conv(sums, self.conv, self.conv_bias, conv_state, ctx.q_starts, ctx.slots, ctx.token_entry, C, xc, silu=True, longest=ctx.longest)
        k.gemm(xc, self.w_x, dbc, EPI_STORE, ctx.gemm_workspace(xc, self.w_x))
        if in_products and k.product_steps_scan(T, C):
            k.scan_product_step(dbc, R, self.w_dt, xc, self.dt_bias, self.A, self.D, sums[:, C:], scan_state, ctx.slots, y)
        else:
            dt = ctx.workspace("mamba.dt", (T, C), torch.float32)
            d = dbc[:, :R]
            k.gemm(d, self.w_dt, dt, EPI_STORE_F32, ctx.gemm_workspace(d, self.w_dt))
            ypart = ctx.workspace("mamba.ypart", (T, C), torch.float32) if N > 64 else None
            need = k.scan_carry_floats(T, ctx.n_entries, ctx.longest, (N + 1) * C)
            carry = ctx.workspace("scan.carry", (need,), torch.float32) if need else None
            k.selective_scan(xc, dbc, R, R + N, dt, self.dt_bias, self.A, self.D, sums[:, C:], scan_state, ctx.q_starts, ctx.slots, y, ypart,
                             ctx.longest, carry)
        k.gemm(y, self.w_o, h, EPI_ACCUM_F32, ctx.gemm_workspace(y, self.w_o))
        ctx.note_left(h, None)


register_mixer("mingru", MinGRU)
register_mixer("mamba1", Mamba1)


class GatedUnit(Mixer):
    graph_safe = True
    SHARPNESS = 8.0             # what r softplus(lambda) is multiplied by: the design fixes it

    def __init__(self, spec, dtype):
        super().__init__(spec, dtype)
        p = spec.params
        self.hidden, self.width, self.blocks, self.taps = int(p["hidden_size"]), int(p["width"]), int(p["blocks"]), int(p["conv"])
        if self.taps < 1:
            raise ValueError("the convolution has at least one tap")
        if self.blocks < 1 or self.width % self.blocks:
            raise ValueError(f"a width of {self.width} does not fall into {self.blocks} equal blocks")
        self.size = self.width // self.blocks
        leaves = _leaves({"y": "y", "y_bias": "y.b", "x": "x", "x_bias": "x.b", "conv": "conv", "conv_bias": "conv.b", "r": "ra", "r_bias": "ra.b",
                          "i": "ri", "i_bias": "ri.b", "lam": "lam", "out": "o"}, p.get("names"))
        self.names = {k: self.name(v) for k, v in leaves.items()}
        self.w_in = self.w_gates = self.w_o = self.conv = self.conv_bias = None
        self.bias_y = self.bias_x = self.bias_r = self.bias_i = self.rate = None
        self.lam = None             # as the file has it (on the host): the kernels read the rate made of it

    def tensors(self):
        n, H, W, B, S = self.names, self.hidden, self.width, self.blocks, self.size
        return {n["y"]: TensorSpec((W, H)), n["y_bias"]: TensorSpec((W,)), n["x"]: TensorSpec((W, H)), n["x_bias"]: TensorSpec((W,)),
                n["conv"]: TensorSpec((W, self.taps), "normal:0.0:0.3"), n["conv_bias"]: TensorSpec((W,)),
                n["r"]: TensorSpec((B, S, S), "normal:0.0:0.1"), n["r_bias"]: TensorSpec((B, S)), n["i"]: TensorSpec((B, S, S), "normal:0.0:0.1"),
                n["i_bias"]: TensorSpec((B, S)), n["lam"]: TensorSpec((W,), "normal:-4.0:1.0"), n["out"]: TensorSpec((H, W))}

    def load(self, tensors, device):
        n = self.names
        get = lambda key: place(tensors[n[key]], device, self.dtype)
        get32 = lambda key: place(tensors[n[key]], device, torch.float32)
        self.w_in = torch.cat([get("y"), get("x")], dim=0).contiguous()             # one product: y | x
        self.w_gates = torch.cat([get("r"), get("i")], dim=1).contiguous()          # a block's two matrices one under the other
        self.w_o = get("out")
        self.conv, self.conv_bias = get32("conv"), get32("conv_bias")
        self.bias_y, self.bias_x = get32("y_bias"), get32("x_bias")
        self.bias_r, self.bias_i = get32("r_bias").reshape(-1), get32("i_bias").reshape(-1)
        self.lam = place(tensors[n["lam"]], "cpu", torch.float32)
        soft = torch.nn.functional.softplus(self.lam.double(), threshold=60.0)
        self.rate = (-self.SHARPNESS * soft).to(torch.float32).to(device)          # once, for every token

    def export(self):
        n, W, S = self.names, self.width, self.size
        w, g = self.w_in.cpu(), self.w_gates.cpu()
        return {n["y"]: w[:W].contiguous(), n["x"]: w[W:].contiguous(), n["r"]: g[:, :S].contiguous(), n["i"]: g[:, S:].contiguous(),
                n["out"]: self.w_o.cpu(), n["conv"]: self.conv.cpu(), n["conv_bias"]: self.conv_bias.cpu(), n["y_bias"]: self.bias_y.cpu(),
                n["x_bias"]: self.bias_x.cpu(), n["r_bias"]: self.bias_r.cpu().view(self.blocks, S), n["i_bias"]: self.bias_i.cpu().view(self.blocks, S),
                n["lam"]: self.lam}

    def step_weight_bytes(self, seen):
        seen.add(self.lam.data_ptr())        # a step reads the rate, not what it was made of
        return super().step_weight_bytes(seen)

    def cache_need(self):
        # one row per request: S [width], then the convolution's last inputs [conv - 1, width]
        return FixedState((self.width * self.taps,), torch.float32)

    def input_weight(self):
        return self.w_in

    def share_input_weight(self, w):
        self.w_in = w

    def forward(self, ctx, x, h, cache, sums=None):
        k = kernels()
        T, W = x.shape[0], self.width
        if sums is None:
            sums = ctx.workspace("unit.sums", (T, 2 * W), torch.float32)
            k.gemm(x, self.w_in, sums, EPI_STORE_F32, ctx.gemm_workspace(x, self.w_in))
        u32 = ctx.workspace("unit.u32", (T, W), torch.float32)
        u = u32 if self.dtype == torch.float32 else ctx.workspace("unit.u", (T, W), self.dtype)
        k.causal_conv(sums[:, W:], self.conv, self.conv_bias, cache.state[:, W:], ctx.q_starts, ctx.slots, ctx.token_entry, W, u,
                      in_bias=self.bias_x, out32=None if u is u32 else u32, longest=ctx.longest)
        gates = ctx.workspace("unit.gates", (T, 2 * W), torch.float32)
        k.head_product(u, self.w_gates, gates)
        out = ctx.workspace("unit.out", (T, W), self.dtype)
        need = k.scan_carry_floats(T, ctx.n_entries, ctx.longest, 2 * W)
        carry = ctx.workspace("scan.carry", (need,), torch.float32) if need else None
        k.gated_unit_scan(u32, gates, self.size, self.bias_r, self.bias_i, self.rate, sums[:, :W], self.bias_y, cache.state, ctx.q_starts, ctx.slots,
                          out, ctx.longest, carry)
        k.gemm(out, self.w_o, h, EPI_ACCUM_F32, ctx.gemm_workspace(out, self.w_o))
        ctx.note_left(h, None)


register_mixer("gated_unit", GatedUnit)
