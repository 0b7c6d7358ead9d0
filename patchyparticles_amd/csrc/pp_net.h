// pp_net.h -- host side of a proposal network (pp_net.cpp, pp_api.cpp).
#pragma once

#include <vector>

#include "pp_internal.h"

struct pp_net {
	int device = 0;
	hipStream_t stream = nullptr;
	ppd::NetDev d{};
	int step = 0;  // Adam steps taken
	// device scratch of host-driven calls and of training batches
	int cap = 0;  // rows (multiple of 32)
	__bf16 *x = nullptr;                                // training samples
	float *xh = nullptr, *y = nullptr, *target = nullptr;  // a caller's rows, their outputs, the targets
	ppd::NetScratch q{};
	// pinned: the gradients (NN_W + NN_B) and the rows' losses of a loss_grad
	// call, which its kernels write straight into host memory
	float *h_out = nullptr, *d_h_out = nullptr;  // host and device address
	int h_cap = 0;                               // rows
	std::vector<void *> allocs;
	~pp_net();
};

namespace ppd {
// grow the scratch of `net` to at least m rows; PP_OK or an error status
int net_reserve(pp_net *net, int m);
}
