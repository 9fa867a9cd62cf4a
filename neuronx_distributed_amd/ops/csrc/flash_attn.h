// The entry points of flash attention that host code calls: flash_attn.hip and
// flash_attn_bwd.hip define them, host/flash_autograd.cpp calls them, and all three
// include this, so that a definition that differs does not compile.
#pragma once
#include <hip/hip_runtime_api.h>

extern "C" {
// st: strides (batch, head, row) of q, k, v, out
void flash_attn_fwd_strided(const void* q, const void* k, const void* v, void* out,
                            void* lse, int B, int Hq, int Hkv, int S, float scale,
                            int causal, int window, const long* st, hipStream_t stream);
// st: of q, k, v, out, dout, dq, dk, dv; dk and dv of Hdk heads, Hkv <= Hdk <= Hq, each
// dividing the next
void flash_attn_bwd_strided(const void* q, const void* k, const void* v, const void* out,
                            const void* dout, const void* lse, void* delta, void* dq,
                            void* dk, void* dv, int B, int Hq, int Hkv, int Hdk, int S,
                            float scale, int causal, int window, const long* st,
                            hipStream_t stream);
// kq, vq (B, Hq, S, 128) summed to Hkv heads; st: of dk, dv
void flash_attn_bwd_reduce(const void* kq, const void* vq, void* dk, void* dv, int B,
                           int Hq, int Hkv, int S, const long* st, hipStream_t stream);
}
