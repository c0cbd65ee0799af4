// CudaQLearning: the reference's tabular Q-learning host class
// (src/q_learning.cuh:8-95), same public signatures, on the HIP engine.
#pragma once
#include <cstddef>
#include <cstdint>
#include <utility>
#include <vector>

struct crl_engine;

class CudaQLearning {
 public:
  // max_mode (additive): 1 = max over the next row seeded with 0, which is what the
  // kernel behind this class upstream computes (update_q_values_kernel,
  // src/kernels.cu:101-110) and therefore the default of the five-argument
  // constructor; 0 = the true max (src/gpu/kernels.cu:35-45, np.max in src/train.py:134),
  // the default of the batched engine and of train().
  CudaQLearning(int width, int height, int action_space_size, float learning_rate = 0.1f,
                float discount_factor = 0.99f, int max_mode = 1);
  ~CudaQLearning();
  CudaQLearning(const CudaQLearning&) = delete;
  CudaQLearning& operator=(const CudaQLearning&) = delete;

  void update_batch(const std::vector<std::pair<int, int>>& states, const std::vector<int>& actions,
                    const std::vector<float>& rewards,
                    const std::vector<std::pair<int, int>>& next_states,
                    const std::vector<bool>& dones);
  // the same from arrays, each with its length
  void update_batch(const std::pair<int, int>* states, size_t batch_size, const int* actions, size_t n_actions,
                    const float* rewards, size_t n_rewards, const std::pair<int, int>* next_states, size_t n_next,
                    const uint8_t* dones, size_t n_dones);
  std::vector<float> get_q_table() const;
  // the same without a copy; valid until the next call that changes the table
  const std::vector<float>& q_values() const { return h_q_table; }
  void set_q_table(const std::vector<float>& q_table);
  int get_best_action(int x, int y) const;
  float get_q_value(int x, int y, int action) const;

 private:
  int width;
  int height;
  int action_space_size;
  float learning_rate;
  float discount_factor;
  std::vector<float> h_q_table;  // host mirror, refreshed after every update
  crl_engine* engine;
  int max_batch_size;
  std::vector<int32_t> batch;  // scratch of update_batch: s, s', a, changed keys
  std::vector<float> changed;  // ... and their new values
};
