// The histogram surrogate network (see surrogate.hip).
#pragma once

#include "engine.hpp"

namespace mlens
{

constexpr int SURR_NIN = 6;        // kappa_tot, shear, smooth fraction, mass-function slope, m_lower, m_upper
constexpr int SURR_PIN = 16;       // inputs padded to one MFMA K step
constexpr int SURR_HIDDEN = 256;
constexpr int SURR_NOUT = 128;     // log10 magnification bins over [-2, 2]
constexpr int SURR_LAYERS = 4;

// where a training pass leaves what the weight gradients read: [feature][row], ld rows each
struct NetTrace
{
	unsigned short* in[SURR_LAYERS];    // a layer's input: the batch, then the hidden activations
	unsigned short* dz16[SURR_LAYERS];  // gradient of its pre-activations in BF16
	float* dz32[SURR_LAYERS];           // and in FP32
	int ld;
};

class Surrogate
{
public:
	Surrogate(int max_batch, uint32_t seed);
	~Surrogate();
	Surrogate(const Surrogate&) = delete;
	Surrogate& operator=(const Surrogate&) = delete;

	size_t num_params() const { return nparams_; }
	void set_params(const float* host);   // FP32 master weights (layer by layer: W [out x in], then b); resets Adam
	void get_params(float* host) const;

	void load_data(const float* x, const float* t, int n);            // x: n x 6 (normalised), t: n x 128 (rows sum to 1)
	double train_step(const int* rows, int m, float lr, float wd);   // one Adam step on rows of the loaded set; mean loss
	double gradients(const float* x, const float* t, int n, float* grads);   // loss and dloss/dparams of one batch (n % 16 == 0)
	void predict(const float* x, int n, float* probs);                // n x 128 softmax outputs
	double time_predict(const float* x, int n, int reps);             // seconds per predicted histogram on the device

	// `steps` of them: step k on rows[k m .. (k + 1) m) at rate lr[k]; losses[k] its mean loss
	void train(const int* rows, int steps, int m, const float* lr, float wd, double* losses);

private:
	NetTrace trace(int M);
	void launch_predict(const unsigned short* x, int rows, float* probs);

	static constexpr int PREDICT_SMALL = 256;   // rows of a request that goes through pinned memory
	static constexpr int PREDICT_ROWS = 8192;   // rows at a time of a larger one

	int max_batch_;
	hipStream_t stream_ = nullptr;
	size_t nparams_ = 0;
	int step_ = 0;
	int ndata_ = 0;
	void* small_ = nullptr;   // pinned: a small request's inputs, then its outputs
	DeviceBuffer<float> w_, g_, m_, v_;
	DeviceBuffer<unsigned short> w16_, wt16_;   // BF16 weights [out x in] and [in x out]
	DeviceBuffer<unsigned short> xall_, xb_, trace16_;
	DeviceBuffer<float> tall_, p_, loss_, trace32_;
	DeviceBuffer<int> idx_;
};

}  // namespace mlens
