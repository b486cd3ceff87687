// What the two files of the native host module share.
#pragma once
#include <Python.h>

#include <ATen/ATen.h>

#include "tdb_attn.h"

// The bound C-ABI entry points.
int (*tdb_host_fixed())(const tdb_fixed_args*, void*);
int (*tdb_host_varlen())(const tdb_varlen_args*, void*);

// Span, delta table (of sequences up to max_len) and per-head tables [.., H, rows, D] of one call; false where no delta table
// for this length is at hand.  No tables: nothing is filled.
bool tdb_host_fill_tables(tdb_pos_args& pos, const at::Tensor* pk, const at::Tensor* pq, int64_t buckets, int64_t max_rel, int64_t max_len, int device);

// Whether somebody records the operations of this thread (a tracer, a dispatch mode): a result made here would be a constant
// to a tracer and nothing at all to a mode.
bool tdb_host_observed();

// A strided tensor of q's device with nothing to record: no gradient (looked at if `grad`), no tangent, no transform wrapped
// around it.
bool tdb_host_plain(const at::Tensor& t, const at::Tensor& q, bool grad);

bool tdb_host_add_encoder(PyObject* module);
