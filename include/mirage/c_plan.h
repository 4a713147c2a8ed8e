/* The plan of a customized operator as the C facade takes it (mirage_graph_customized). */
#pragma once

typedef struct mirage_c_plan {
  int grid_dim[3];
  int block_dim[3];
  int forloop_range;
  int reduction_dimx;
  int num_inputs;
  int input_map[4][3];
  int forloop_dim[4];
  int input_smem_layout[4];
  int output_map[3];
  int num_ops;
  int op_type[16];
  int op_num_operands[16];
  int op_operands[16][2][2];
} mirage_c_plan;
