// The vLLM cache layout (cache_engine.rs:81-100) as the kernels that write it see it.
#pragma once

#include "common.h"
#include "device_types.h"

namespace hipattn {

struct CacheGeom {
  int64_t num_blocks;
  int num_heads;
  int head_size;
  int block_size;
  int x;
  int64_t k_block_stride, k_head_stride;  // elements
  int64_t v_block_stride, v_head_stride;
};

// Block and offset of a slot; block -1: not cached (negative, or past the cache).
__device__ __forceinline__ int64_t slot_block(int64_t slot, const CacheGeom &g, int &off) {
  int64_t blk = -1;
  off = 0;
  if (slot >= 0 && slot <= 0x7fffffff) {  // (a 64-bit division is some hundred instructions in front of every store)
    const unsigned b = (unsigned)slot / (unsigned)g.block_size;
    off = (int)((unsigned)slot - b * (unsigned)g.block_size);
    blk = b;
  } else if (slot >= 0) {
    blk = slot / g.block_size;
    off = (int)(slot % g.block_size);
  }
  return blk < g.num_blocks ? blk : -1;
}

inline CacheGeom cache_geometry(const hipattn_tensor *key_cache, const hipattn_tensor *value_cache,
                         const char *op) {
  check_tensor(key_cache, "key_cache", 5);
  check_tensor(value_cache, "value_cache", 4);
  HA_CHECK(is_float_dtype(key_cache->dtype), "%s: key_cache must be a float type", op);
  HA_CHECK(key_cache->dtype == value_cache->dtype, "%s: key_cache/value_cache dtype mismatch", op);
  CacheGeom g;
  g.num_blocks = key_cache->sizes[0];
  g.num_heads = (int)key_cache->sizes[1];
  g.block_size = (int)key_cache->sizes[3];
  g.x = (int)key_cache->sizes[4];
  g.head_size = (int)(key_cache->sizes[2] * key_cache->sizes[4]);
  HA_CHECK(g.x == 16 / dtype_size(key_cache->dtype),
           "%s: key_cache last dim must be 16/sizeof(dtype) = %d, got %d", op,
           16 / dtype_size(key_cache->dtype), g.x);
  HA_CHECK(value_cache->sizes[0] == g.num_blocks && value_cache->sizes[1] == g.num_heads &&
               value_cache->sizes[2] == g.head_size && value_cache->sizes[3] == g.block_size,
           "%s: value_cache shape does not match key_cache", op);
  HA_CHECK(key_cache->strides[4] == 1 && key_cache->strides[3] == g.x &&
               key_cache->strides[2] == (int64_t)g.x * g.block_size,
           "%s: key_cache inner dims must be contiguous", op);
  HA_CHECK(value_cache->strides[3] == 1 && value_cache->strides[2] == g.block_size,
           "%s: value_cache inner dims must be contiguous", op);
  g.k_block_stride = key_cache->strides[0];
  g.k_head_stride = key_cache->strides[1];
  g.v_block_stride = value_cache->strides[0];
  g.v_head_stride = value_cache->strides[1];
  check_data(key_cache, "key_cache");
  check_data(value_cache, "value_cache");
  return g;
}

}  // namespace hipattn
