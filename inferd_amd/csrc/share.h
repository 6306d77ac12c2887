// The K-shares of a GEMM's last tiles (gemm_w.hip, gemm_n.hip): rem tiles of G units each are shared out evenly among
// blocks 0 .. n - 1 (rem < n), so that no CU waits for a partly filled last round. Block b's share starts at unit
// share_start(b); unit u lies in the share of block share_of(u). A share is shorter than a tile, so it is part of at
// most two, and of each it sums one piece. The pieces in order are numbered by block where every tile is cut at the
// same units (n a multiple of rem), else by block + tile. 32-bit arithmetic, (rem G + 1) n < 2^32: n is at most the CU
// count, and with activations and weights below 2 GiB each (the launchers' bound) rem G stays below 3 million at 256 CUs.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ifd {

__host__ __device__ inline int share_start(int b, int rem, int n, int G) { return (int)((uint32_t)b * rem * G / n); }
__host__ __device__ inline int share_of(int u, int rem, int n, int G) {
  return (int)(((uint32_t)u * n + n - 1) / ((uint32_t)rem * G));
}
__host__ __device__ inline int share_piece(int b, int tile, int rem, int n) { return n % rem ? b + tile : b; }
__host__ __device__ inline int share_pieces(int rem, int n) { return rem == 0 ? 0 : n % rem ? n + rem - 1 : n; }

}  // namespace ifd
