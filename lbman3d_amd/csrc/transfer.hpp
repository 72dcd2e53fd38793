// transfer.hpp — fields between host arrays (FP64) and a handle's device
// arrays (transfer.hip). Every call returns when its host arrays are read or
// written.
#pragma once

#include "solver_state.hpp"

namespace lbm {

constexpr int kMaxItems = 16;

// One array of V values: host = base + device value.
struct FetchItem {
    const void* dev;
    double* host;
    double base;
};
// One array of V values: device = host value - base.
struct PutItem {
    void* dev;
    const double* host;
    double base;
};
int fetch_fields(lbm_solver* s, const FetchItem* items, int count);
int put_fields(lbm_solver* s, const PutItem* items, int count);
// The fields given (any may be null), then populations Feq(rho, u).
int put_state(lbm_solver* s, const double* rho, const double* const u[3], const double* q);
// rho = rho0 and populations Feq(rho0, u).
int put_rest(lbm_solver* s);

// Order parameter and director of every cell, [V] and [V][3].
int fetch_order_director(lbm_solver* s, double* order, double* director);

// The pinned buffers live while a handle does.
void staging_open();
void staging_close();

}  // namespace lbm
