// Flash attention as a native autograd function: what _FlashAttnFn of ops/__init__.py
// does, without the interpreter in either direction.  Short sequences wait for their
// host: forward and backward of 241 tokens, 32 heads, are 42 us of kernels, and a pass
// took 157 us, now 103; 3 x 617 of 32/8 heads 169, now 111; from about 1200 tokens on
// the kernels last longer.  What is left is the engine's own thread (an empty function
// takes 74 in Python, a native product 53) and the launches.
//
// Host code only; the kernels are libnxd_ops.so's.

#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>

#include "../flash_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// as _fa_ok_layout: rows of whole 16-byte words, 31 of them less than 2 GB
bool good_layout(const Tensor& t) {
  if (t.stride(3) != 1 || t.stride(2) >= 1 << 25) return false;
  for (int i = 0; i < 3; ++i)
    if (t.stride(i) & 7) {
      for (int j = 0; j < 3; ++j)
        if (t.size(j) > 1 && t.stride(j) & 7) return false;
      break;
    }
  return true;
}

Tensor operand(const Tensor& t) {
  Tensor x = good_layout(t) ? t : t.contiguous();
  return (size_t)x.data_ptr() & 15 ? x.clone() : x;
}

// an empty tensor in the layout of t
Tensor alloc_like(const Tensor& t) {
  const auto B = t.size(0), H = t.size(1), S = t.size(2), D = t.size(3);
  if (t.stride(1) == D && t.stride(2) == H * D)
    return at::empty({B, S, H, D}, t.options()).permute({0, 2, 1, 3});
  return at::empty({B, H, S, D}, t.options());
}

long* strides(long* at, const Tensor& t) {
  for (int i = 0; i < 3; ++i) *at++ = t.stride(i);
  return at;
}

struct FlashAttention : torch::autograd::Function<FlashAttention> {
  // heads: of dK and dV that the backward's kernel writes
  static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_,
                        const Tensor& v_, bool causal, double scale, int64_t window,
                        int64_t heads) {
    const Tensor q = operand(q_), k = operand(k_), v = operand(v_);
    const int B = q.size(0), Hq = q.size(1), S = q.size(2), Hkv = k.size(1);
    Tensor out = alloc_like(q);
    Tensor lse = at::empty({B, Hq, S}, q.options().dtype(at::kFloat));
    long st[12];
    strides(strides(strides(strides(st, q), k), v), out);
    flash_attn_fwd_strided(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                           lse.data_ptr(), B, Hq, Hkv, S, (float)scale, causal,
                           (int)window, st, c10::hip::getCurrentHIPStream());
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["how"] = std::vector<int64_t>{causal, window, heads};
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3],
                 &lse = saved[4];
    const auto how = ctx->saved_data["how"].toIntVector();
    const float scale = (float)ctx->saved_data["scale"].toDouble();
    const int B = q.size(0), Hq = q.size(1), S = q.size(2), D = q.size(3);
    const int Hkv = k.size(1), heads = (int)how[2];
    const Tensor dout = operand(grads[0]);
    Tensor delta = at::empty({B, Hq, S}, lse.options());
    Tensor dq = alloc_like(q);
    Tensor dk = alloc_like(k), dv = alloc_like(v), dk_pq = dk, dv_pq = dv;
    if (heads != Hkv) {                  // then summed over the heads of a group
      dk_pq = at::empty({B, heads, S, D}, k.options());
      dv_pq = at::empty({B, heads, S, D}, v.options());
    }
    long st[24], *at = st;
    for (const Tensor* t : {&q, &k, &v, &out, &dout, (const Tensor*)&dq,
                            (const Tensor*)&dk_pq, (const Tensor*)&dv_pq})
      at = strides(at, *t);
    const hipStream_t stream = c10::hip::getCurrentHIPStream();
    flash_attn_bwd_strided(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                           dout.data_ptr(), lse.data_ptr(), delta.data_ptr(),
                           dq.data_ptr(), dk_pq.data_ptr(), dv_pq.data_ptr(), B, Hq, Hkv,
                           heads, S, scale, (int)how[0], (int)how[1], st, stream);
    if (heads != Hkv) {
      strides(strides(st, dk), dv);
      flash_attn_bwd_reduce(dk_pq.data_ptr(), dv_pq.data_ptr(), dk.data_ptr(),
                            dv.data_ptr(), B, heads, Hkv, S, st, stream);
    }
    return {dq, dk, dv, {}, {}, {}, {}};
  }
};

Tensor flash_attention(const Tensor& q, const Tensor& k, const Tensor& v, bool causal,
                       double scale, int64_t window, int64_t heads) {
  return FlashAttention::apply(q, k, v, causal, scale, window, heads);
}

}  // namespace

TORCH_LIBRARY(nxd_host, m) {
  m.def("flash_attention(Tensor q, Tensor k, Tensor v, bool causal, float scale, "
        "int window, int heads) -> Tensor",
        torch::dispatch(c10::DispatchKey::CompositeImplicitAutograd,
                        TORCH_FN(flash_attention)));
}
