// attn_split.h -- the context-split decode attention (attn_split.hip) for the
// C-ABI entry points of attn.hip, which check the arguments.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace mxh {
// Bytes of the records at the workspace's front (a multiple of 16; from 4097
// positions on the workspace has room for q bf16 (M, Hq, 128) after them).
size_t attn_split_record_bytes(int M, int Hq, int Hkv, int max_pos);
// q bf16 (M, Hq, 128), kvk / kvv 16- and 4-byte aligned, G = Hq / Hkv a power of
// two up to 16; workspace of mxfp4_attn_decode_workspace_size bytes.
int attn_split(const void* q, const uint8_t* kvk, const uint8_t* kvv, const int32_t* dpos, float* sc, float* o,
               uint8_t* oq, uint8_t* os, int M, int Hq, int Hkv, int max_pos, void* workspace, hipStream_t st);
}  // namespace mxh
