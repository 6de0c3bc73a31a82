// Arguments and launcher of the fp32 / fp64 GEMM chain kernels (gemm_chain_f32.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ditto {

struct F32ChainArgs {
  const void* a;  // float or double (f64)
  const void* b;
  const void* c;
  void* f;
  long long a_bs, b_bs, c_bs, f_bs;  // batch strides, elements
  int a_rs, b_rs, c_rs, f_rs;        // row strides, elements
  int M, N, K, L, batch;
  int mblocks;    // workgroups per batch entry
  int row_tiles;  // fp32: rows of a workgroup / 16 (1 or 2); fp64: workgroups own 32 rows
  int width;      // fp32: columns of F a workgroup owns: 0 (all), 64, 32 or 16
  int col_blocks; // fp32: workgroups that share out the columns of a block of rows
  int b_lk;     // B stored [L][K]
  int relu;
  int relu_out;  // ReLU on the output
  int softmax;   // inter path: softmax over L of scale * (A.B)
  float softmax_scale;
  int f64;       // elements are doubles
  unsigned block0;  // fp32: workgroups in front of this launch's (filled by the launcher)
};

int f32_chain_lds_bytes_host(int K, int N, int f64, int row_tiles, int width);
int f32_chain_width(int K, int N, long long row_blocks, int cus);
bool f32_chain_exact(int K, int N, long long strides);  // whole tiles of columns and rows in 16-byte pieces; the strides ORed together
int f32_chain_max_dim();  // largest K and N the kernels take
hipError_t launch_gemm_chain_f32(const F32ChainArgs& args, hipStream_t stream);

}  // namespace ditto
