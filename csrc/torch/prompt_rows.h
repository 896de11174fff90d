// What the module of attention_autograd.cpp takes from prompt_rows.cpp
#pragma once
#include <Python.h>

PyObject* kca_few_rows(PyObject*, PyObject* const*, Py_ssize_t);
PyObject* kca_norm_rows(PyObject*, PyObject* const*, Py_ssize_t);
PyObject* kca_rope_rows(PyObject*, PyObject* const*, Py_ssize_t);
PyObject* kca_packed_rows(PyObject*, PyObject* const*, Py_ssize_t);
PyObject* kca_init_rows(PyObject*, PyObject* const*, Py_ssize_t);
